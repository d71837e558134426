// Shared parts of the matrix-core GEMMs whose tiles stream global -> LDS
// through a ring of stages: wait counts, the ring's barrier, the XCD-grouped
// tile order and the host's launch helpers.
#pragma once

#include <atomic>
#include <mutex>
#include <set>
#include <utility>

#include "device_utils.hpp"

namespace mrt {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// s_waitcnt immediate waiting for vmcnt <= n (expcnt and lgkmcnt left alone).
constexpr int vm_wait_imm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }

// Workgroup barrier of the global -> LDS rings: every LDS read this wave has
// issued has returned (so another wave may refill that stage after the
// barrier), then the waves meet.  Unlike __syncthreads() it does not wait for
// this wave's loads still in flight to later stages (a release fence would
// wait for every outstanding LDS write, direct-to-LDS loads included): the
// stage about to be read is awaited with an explicit vmcnt before it.  The
// asm is a compiler barrier for memory operations.
__device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Tile of block L of a 1-D grid in the XCD-grouped order: blocks are dealt to
// the 8 XCDs in turn (L % 8), each XCD takes a contiguous range of tile ids,
// and tile ids run down GM row tiles before the next column tile, so the
// blocks that one XCD runs together share GM A tiles and a few B tiles in its
// L2.  A bijection of [0, tm * tn).
__device__ __forceinline__ void grouped_tile(int L, int tm, int tn, int GM, int& mt, int& nt) {
  const int tiles = tm * tn, x = L & 7, q = tiles >> 3, rem = tiles & 7;
  const int pid = x * q + min(x, rem) + (L >> 3);
  const int g = pid / (GM * tn), first = g * GM, gsz = min(tm - first, GM);
  const int w = pid - g * GM * tn;
  mt = first + w % gsz;
  nt = w / gsz;
}

// Dynamic LDS above 64 KB needs an explicit allowance, once per kernel and device.
inline void allow_dynamic_lds(const void* fn, size_t bytes) {
  static std::mutex mu;
  static std::set<std::pair<const void*, int>> done;
  int dev = 0;
  MRT_HIP_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> g(mu);
  if (done.count({fn, dev})) return;
  MRT_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
  done.insert({fn, dev});
}

// Compute units of the current device (cached per device).
inline int device_cus() {
  constexpr int kMaxDev = 64;
  static std::atomic<int> cache[kMaxDev] = {};
  int dev = 0;
  MRT_HIP_CHECK(hipGetDevice(&dev));
  int v = (dev >= 0 && dev < kMaxDev) ? cache[dev].load(std::memory_order_relaxed) : 0;
  if (v == 0) {
    MRT_HIP_CHECK(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev));
    if (dev >= 0 && dev < kMaxDev) cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

}  // namespace mrt
