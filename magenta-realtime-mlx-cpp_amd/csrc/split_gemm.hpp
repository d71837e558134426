// fp32 products on the bf16 matrix cores.  A float is the exact sum of three
// bf16 parts (8 significant bits each, rounded to nearest: part 2 at most 2^-9,
// part 3 at most 2^-18 of the value), so a product of two floats is nine bf16
// products, of which the three smallest together stay below 2^-25 of it: six
// v_mfma_f32_32x32x16_bf16 per 16-deep step, accumulated in fp32, the smallest
// first, compute the fp32 product sum.  Six bf16 products cost 192 cycles of a
// SIMD per 32 x 32 x 16 step, the fp32 instruction 512: 2.7 times its rate, with
// fewer roundings of the accumulator (measured errors against 64 bits: no
// larger than the fp32 instruction's or a chain of fused multiply-adds').
//
// Operands are stored split: row r of K values (K % 32 == 0) is K / 32 groups of
// 32 values, each group its 32 first parts, 32 second parts, 32 third parts:
// 192 bytes (split_index).
#pragma once

#include "mfma_ring.hpp"

namespace mrt {

constexpr int kSplitGroup = 96;  // bf16 values of 32 split floats

// Offset of part 0 of element k of row r (K values a row); part p: + 32 p.
__host__ __device__ inline size_t split_index(size_t r, int k, int K) {
  return (r * (size_t)(K >> 5) + (k >> 5)) * kSplitGroup + (k & 31);
}

// The parts of a float.  A value that rounds up to infinity keeps a truncated
// first part; infinities and NaN are their first part alone.
__device__ __forceinline__ void split3(float a, bf16 (&p)[3]) {
  p[0] = f2bf(a);
  if ((p[0] & 0x7fff) == 0x7f80) p[0] = (bf16)(__float_as_uint(a) >> 16);
  float r = a - bf2f(p[0]);
  r = r == r ? r : 0.f;
  p[1] = f2bf(r);
  p[2] = f2bf(r - bf2f(p[1]));
}

__device__ __forceinline__ void store_split(bf16* base, size_t idx, float v) {
  bf16 p[3];
  split3(v, p);
  base[idx] = p[0];
  base[idx + 32] = p[1];
  base[idx + 64] = p[2];
}

// Four consecutive elements (k % 4 == 0).
__device__ __forceinline__ void store_split4(bf16* base, size_t idx, const float (&v)[4]) {
  bf16 p[4][3];
#pragma unroll
  for (int e = 0; e < 4; ++e) split3(v[e], p[e]);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    uint2 w;
    w.x = (uint32_t)p[0][q] | ((uint32_t)p[1][q] << 16);
    w.y = (uint32_t)p[2][q] | ((uint32_t)p[3][q] << 16);
    *reinterpret_cast<uint2*>(base + idx + 32 * q) = w;
  }
}

// The multiply loop of a BM x BN tile, WM x WN waves, an S-stage ring of
// 32-deep k-tiles (one 192-byte group of every A and B row).  A row is 12
// chunks of 16 bytes; chunk c of row r is stored at chunk (c + (r / 4) % 4) % 12:
// 16 consecutive rows at a pitch of 12 chunks then hit the 16 chunk banks once.
// The matrix cores bound it (48 products, 1,536 cycles, per 24 LDS reads of a
// 64 x 64 wave tile).
template <int BM, int BN, int WM, int WN, int S>
struct SplitTile {
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int MI = BM / WM / 32, NJ = BN / WN / 32;
  static constexpr int kStage = (BM + BN) * 192;
  static constexpr int LA = BM * 12 / kThreads, LB = BN * 12 / kThreads;  // loads per thread and k-tile
  static constexpr size_t kLds = (size_t)S * kStage;
  static_assert(BM * 12 % kThreads == 0 && BN * 12 % kThreads == 0, "whole loads per wave");
  static_assert(kLds <= 160 * 1024 && (S - 2) * (LA + LB) < 64, "LDS of one CU, vmcnt range");

  // row and source chunk of load q of this thread
  __device__ static void load_pos(int q, int& row, int& chunk) {
    const int idx = (q * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 64 + (threadIdx.x & 63);
    row = idx / 12;
    const int pos = idx - row * 12, c = pos - ((row >> 2) & 3);
    chunk = c < 0 ? c + 12 : c;
  }

  // k-tiles kb .. ke - 1; point(kt, ap, bp) sets this thread's source pointers
  // of k-tile kt (chunk included).
  template <class Point>
  __device__ static void run(unsigned char* lds, int kb, int ke, Point&& point, f32x16_t (&acc)[MI][NJ]) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid / WN, wn = wid % WN;
    const bf16* ap[LA];
    const bf16* bp[LB];
    int slot = 0;  // ring stage of the next issue
    auto issue = [&](int kt) {
      point(min(kt, ke - 1), ap, bp);  // past the end: the last tile again, into a free stage
      unsigned char* st = lds + slot * kStage;
      slot = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
      for (int q = 0; q < LA; ++q)
        __builtin_amdgcn_global_load_lds((const MRT_GLOBAL void*)ap[q], (MRT_LDS void*)(st + (q * kWaves + wid) * 1024),
                                         16, 0, 0);
#pragma unroll
      for (int q = 0; q < LB; ++q)
        __builtin_amdgcn_global_load_lds((const MRT_GLOBAL void*)bp[q],
                                         (MRT_LDS void*)(st + BM * 192 + (q * kWaves + wid) * 1024), 16, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll
    for (int t = 0; t < S - 1; ++t) issue(kb + t);
    const int lr = lane & 31, lh = lane >> 5;
    int rd = 0;  // ring stage to read
    for (int kt = kb; kt < ke; ++kt) {
      __builtin_amdgcn_s_waitcnt(vm_wait_imm((S - 2) * (LA + LB)));  // this wave's loads of tile kt have landed
      ring_barrier();  // every wave's loads of tile kt; every wave is done with tile kt - 1
      issue(kt + S - 1);
      const unsigned char* st = lds + rd * kStage;
      rd = rd + 1 == S ? 0 : rd + 1;
      v8 a[2][MI][3], b[2][NJ][3];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const int r = wm * (BM / WM) + i * 32 + lr;
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            int c = 4 * p + 2 * s + lh + ((r >> 2) & 3);
            c = c >= 12 ? c - 12 : c;
            a[s][i][p] = *reinterpret_cast<const v8*>(st + r * 192 + c * 16);
          }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int r = wn * (BN / WN) + j * 32 + lr;
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            int c = 4 * p + 2 * s + lh + ((r >> 2) & 3);
            c = c >= 12 ? c - 12 : c;
            b[s][j][p] = *reinterpret_cast<const v8*>(st + BM * 192 + r * 192 + c * 16);
          }
        }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};  // smallest products first
#pragma unroll
        for (int u = 0; u < 6; ++u)
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][i][pa[u]], b[s][j][pb[u]], acc[i][j], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_waitcnt(vm_wait_imm(0));  // no copy into LDS outlives the block
  }
};

// W (N, K) fp32 -> split rows (split_kernels.hip).
void split_rows(const float* W, long N, int K, bf16* out, hipStream_t s);

}  // namespace mrt
