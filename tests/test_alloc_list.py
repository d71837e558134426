"""A model's allocations, compiled for the CPU.

  * The list takes additions from several threads (under the thread sanitizer): the
    parts built on first use are built on whichever thread comes first, and distinct
    states of one model may be driven from distinct threads.
  * A group of allocations is kept as a whole, or given back as a whole where there
    is no memory for one of them (the caller then goes without that part) or where
    building throws.
"""

from __future__ import annotations

import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "magenta-realtime-mlx-cpp_amd" / "csrc"

THREADS = r"""
#include <cstdint>
#include <set>
#include <thread>
#include "alloc_list.hpp"
int main() {
  constexpr int kThreads = 4, kEach = 5000;
  mrt::AllocList list;
  std::vector<std::thread> th;
  for (int t = 0; t < kThreads; ++t)
    th.emplace_back([&, t] {
      for (int i = 0; i < kEach; ++i) {
        auto p = [&](int k) { return reinterpret_cast<void*>(static_cast<uintptr_t>((t * kEach + i) * 3 + k + 1)); };
        list.add(p(0));
        list.add(std::vector<void*>{p(1), p(2)});
      }
    });
  for (auto& t : th) t.join();
  std::set<void*> once;
  long n = 0;
  list.drain([&](void* p) { once.insert(p); ++n; });
  list.drain([&](void*) { ++n; });
  return n == 3l * kThreads * kEach && (long)once.size() == n ? 0 : 1;
}
"""


GROUPS = r"""
#include <set>
#include <stdexcept>
#include "alloc_list.hpp"
struct Dev {
  std::set<void*>* live;
  int* left;  // allocations that there is memory for
  int* syncs;
  bool alloc(void** p, size_t bytes) const {
    if (bytes == 0) throw std::runtime_error("other error");
    if (*left == 0) return false;
    --*left;
    *p = new char[bytes];
    live->insert(*p);
    return true;
  }
  void free(void* p) const {
    if (live->erase(p) != 1) throw std::runtime_error("freed twice");
    delete[] static_cast<char*>(p);
  }
  void sync() const { ++*syncs; }
};
int main() {
  std::set<void*> live;
  int left = 0, syncs = 0;
  const Dev dev{&live, &left, &syncs};
  mrt::AllocList list;
  for (int room = 0; room <= 3; ++room) {  // three allocations, memory for `room` of them
    left = room;
    mrt::AllocGroup<Dev> g(dev);
    int got = 0;
    for (int i = 0; i < 3; ++i) got += g.alloc(8) != nullptr;
    if (got != room) return 1;
    left = 9;  // memory again does not mend the group
    if (room < 3 && g.alloc(8) != nullptr) return 2;
    if (g.keep(list) != (room == 3)) return 3;
    if (live.size() != (room == 3 ? 3u : 0u) || syncs != room + 1) return 4;
  }
  left = 2;
  try {  // a build that throws gives its allocations back, after the work that writes them
    mrt::AllocGroup<Dev> g(dev);
    g.alloc(8);
    g.alloc(0);
    return 5;
  } catch (const std::runtime_error&) {
  }
  if (live.size() != 3 || syncs != 5) return 6;
  list.drain([&](void* p) { dev.free(p); });
  return live.empty() ? 0 : 7;
}
"""


def run(tmp_path, program, *flags):
    src, exe = tmp_path / "allocs.cpp", tmp_path / "allocs"
    src.write_text(program)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", *flags, f"-I{CSRC}", str(src), "-o", str(exe), "-lpthread"],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout + r.stderr)


def test_allocations_added_from_several_threads(tmp_path):
    run(tmp_path, THREADS, "-fsanitize=thread")


def test_groups_are_kept_or_given_back(tmp_path):
    run(tmp_path, GROUPS, "-fsanitize=address")


def test_model_keeps_its_allocations_in_the_list():
    header = (CSRC / "model.hpp").read_text()
    model = header[header.index("class Model {"):header.index("struct EncoderBufs")]
    assert "AllocList allocs_;" in model and "std::vector<void*>" not in model
