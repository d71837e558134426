// fp32 products on the bf16 matrix cores.  A float is the exact sum of three
// bf16 parts (8 significant bits each, rounded to nearest: part 2 at most 2^-9,
// part 3 at most 2^-18 of the value), so a product of two floats is nine bf16
// products, of which the three smallest together stay below 2^-25 of it: six
// v_mfma_f32_32x32x16_bf16 per 16-deep step, accumulated in fp32, compute the
// fp32 product sum.  Six bf16 products cost 192 cycles of a SIMD per 32 x 32 x 16
// step, the fp32 instruction 512: 2.7 times its rate.
//
// The instruction rounds its accumulator several times over its 16 terms, so the
// five small products have a sum of their own where the registers allow
// (CoreSplitFine): the errors against 64 bits are then below those of the fp32
// instruction and of a chain of fused multiply-adds (fp32 encoder of 64 .. 1006
// ids 0.56e-6 .. 4.9e-6 against 1.3e-6 .. 5.1e-6 of the chain; a temporal step after
// it 0.39e-6 .. 0.60e-6 against 0.62e-6).  In one sum they are as large in the
// encoder and twice as large after the cross attention (1.2e-6), whose mean over
// the keys takes away what differs from key to key: the roundings of one sum do not.
//
// Operands are stored split: row r of K values (K % 32 == 0) is K / 32 groups of
// 32 values, each group its 32 first parts, 32 second parts, 32 third parts:
// 192 bytes (split_index).
#pragma once

#include "ring_gemm.hpp"

namespace mrt {

constexpr int kSplitGroup = 96;  // bf16 values of 32 split floats

// Offset of part 0 of element k of row r (K values a row); part p: + 32 p.
__host__ __device__ inline size_t split_index(size_t r, int k, int K) {
  return (r * (size_t)(K >> 5) + (k >> 5)) * kSplitGroup + (k & 31);
}

// The parts of a float: exact for values of at least 2^-110 (below, bits under
// bf16's smallest subnormal, 2^-133, are lost).  A value that rounds up to infinity
// keeps a truncated first part; infinities and NaN are their first part alone
// (resum_not_finite has their products).
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

// Split operands in the GEMM ring: a k-tile is 32 deep, a row of it one 192-byte
// group of 12 chunks of 16 bytes; chunk c of row r is stored at chunk
// (c + (r / 4) % 4) % 12: 16 consecutive rows at a pitch of 12 chunks then hit the
// 16 chunk banks once.  The matrix cores bound it (24 products, 768 cycles, per
// 12 LDS reads of a 64 x 64 wave tile's 16-deep step).
struct CoreSplit {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static constexpr int kChunks = 12, kSteps = 2, kParts = 3, kDepth = 32;
  static constexpr int kProducts = 6;
  static constexpr bool kFine = false;
  __device__ static int place(int r, int chunk) {
    const int c = chunk + ((r >> 2) & 3);
    return c >= 12 ? c - 12 : c;
  }
  __device__ static int chunk_at(int r, int pos) {
    const int c = pos - ((r >> 2) & 3);
    return c < 0 ? c + 12 : c;
  }
  __device__ static int chunk(int step, int part, int half) { return 4 * part + 2 * step + half; }
  // product u of six, the smallest first
  __device__ __forceinline__ static void mma(const v8 (&a)[3], const v8 (&b)[3], int u, f32x16_t& c) {
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[pb[u]], a[pa[u]], c, 0, 0, 0);
  }
};

// The same with the five small products summed apart from the largest, so that the
// whole sum meets one instruction per 16 terms instead of six (the same time: the
// fp32 encoder 5.79 and 5.82 ms).
struct CoreSplitFine : CoreSplit {
  static constexpr bool kFine = true;
};

// sum + the products of `groups` groups of two split rows, as fused multiply-adds of
// the whole floats; NaN as soon as the sum is.
__device__ inline float split_dot(const bf16* a, const bf16* b, int groups, float sum) {
  for (int g = 0; g < groups && sum == sum; ++g, a += kSplitGroup, b += kSplitGroup)
    for (int e = 0; e < 32; e += 8) {
      uint4 u[3], v[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        u[p] = ld_g16(a + 32 * p + e);
        v[p] = ld_g16(b + 32 * p + e);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        auto whole = [&](const uint4 (&q)[3]) {
          return (bf2f(reinterpret_cast<const bf16*>(&q[0])[k]) + bf2f(reinterpret_cast<const bf16*>(&q[1])[k])) +
                 bf2f(reinterpret_cast<const bf16*>(&q[2])[k]);
        };
        sum = fmaf(whole(u), whole(v), sum);
      }
    }
  return sum;
}

// An infinity times the other operand's small parts, zeros or of the other sign, is
// NaN where the float product is infinite.  So sums that are not finite are taken
// again as plain fp32 sums: sum_of(row, column of the tile).  A product and an add per
// sum look for them; where there are some, those take the vector ALUs' time (51 codec
// frames of nothing but NaN, whose sums end early: 43 ms against 2.7).
template <class Tile, class F>
__device__ __forceinline__ void resum_not_finite(typename Tile::State& s, F&& sum_of) {
  constexpr int kSums = Tile::MI * Tile::NJ * 16;
  float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < kSums; ++e) t[e & 3] = fmaf(s.acc[e / 16 / Tile::NJ][e / 16 % Tile::NJ][e % 16], 0.f, t[e & 3]);
  t[0] = (t[0] + t[1]) + (t[2] + t[3]);
  if (__builtin_expect(__ballot(t[0] != t[0]) == 0, true)) return;
#pragma unroll 1
  for (int e = 0; e < kSums; ++e) {
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < kSums; ++q) v = q == e ? s.acc[q / 16 / Tile::NJ][q / 16 % Tile::NJ][q % 16] : v;
    if (fabsf(v) < INFINITY) continue;
    int row, col;
    Tile::sum_pos(e, row, col);
    v = sum_of(row, col);
#pragma unroll
    for (int q = 0; q < kSums; ++q) {
      float& c = reinterpret_cast<float*>(&s.acc[q / 16 / Tile::NJ][q / 16 % Tile::NJ])[q % 16];
      c = q == e ? v : c;
    }
  }
}

// W (N, K) fp32 -> split rows (split_kernels.hip).
void split_rows(const float* W, long N, int K, bf16* out, hipStream_t s);

}  // namespace mrt
