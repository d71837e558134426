"""The list of a model's allocations takes additions from several threads: the
parts built on first use are built on whichever thread comes first, and distinct
states of one model may be driven from distinct threads.  The list is compiled
for the CPU under the thread sanitizer."""

from __future__ import annotations

import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "magenta-realtime-mlx-cpp_amd" / "csrc"

PROGRAM = r"""
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


def test_allocations_added_from_several_threads(tmp_path):
    src, exe = tmp_path / "alloc_list.cpp", tmp_path / "alloc_list"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", f"-I{CSRC}", str(src), "-o", str(exe),
                    "-lpthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_model_keeps_its_allocations_in_the_list():
    header = (CSRC / "model.hpp").read_text()
    model = header[header.index("class Model {"):header.index("struct EncoderBufs")]
    assert "AllocList allocs_;" in model and "std::vector<void*>" not in model
