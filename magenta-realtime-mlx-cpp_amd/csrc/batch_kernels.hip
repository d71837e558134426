// Batched-stream decode kernels for gfx950: B independent streams decoded
// together, R = 2B activation rows (both CFG rows of every stream), R <= 64.
//
// At R = 64 every weight row meets 64 activation rows, so the projections are
// skinny GEMMs and run on the matrix cores: v_mfma_f32_16x16x32_{bf16,f16}, one
// block per 16 output columns, the 8 waves of a block splitting K and summing
// their partial tiles through LDS in a fixed order (deterministic).  The
// activations (R x K, at most 360 KB) are read by every block from L2; the
// weights stream from HBM/MALL once per step.  Both are kept in fragment order
// (batch.hpp), so an operand load of a wave is 1 KB of consecutive addresses.
#include <algorithm>
#include <type_traits>

#include "batch.hpp"
#include "device_utils.hpp"
#include "kernels.hpp"
#include "mfma_ring.hpp"

namespace mrt {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// The 16x16x32 matrix instruction of each 16-bit storage type.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<bf16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  __device__ __forceinline__ static f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};
template <>
struct Mfma16<f16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  __device__ __forceinline__ static f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};

constexpr int kBgCols = 16;  // output columns per block
constexpr int kBgWaves = 8;  // waves per block, splitting K
constexpr int kBgThreads = 64 * kBgWaves;

// ---- epilogues: op(m, n, v[P]) with v the fp32 sums of output (m, n) ---------------

template <typename T>
struct BStore {
  T* y;
  int ldy;
  __device__ void operator()(int m, int n, const float (&v)[1]) const { y[(size_t)m * ldy + n] = St<T>::st(v[0]); }
};

template <typename T>
struct BF32 {
  float* y;
  int ldy;
  __device__ void operator()(int m, int n, const float (&v)[1]) const { y[(size_t)m * ldy + n] = St<T>::rnd(v[0]); }
};

// Residual update; the residual values are read at the start of the kernel
// (pre), so the epilogue does not wait for them.  The updated rows are written
// to r and, in fragment order, to rf; the sum of squares of each updated row
// over the block's 16 columns goes to ssq[m * (N / 16) + tile], the partials a
// normalised consumer reads (BNorm).
template <typename T>
struct BResid {
  T* r;
  int ldr;
  T* rf;
  float* ssq;
  static constexpr bool kPre = true;
  __device__ float pre(int m, int n) const { return St<T>::ld(r[(size_t)m * ldr + n]); }
  __device__ float operator()(int m, int n, const float (&v)[1], float x) const {
    const T y = St<T>::st(x + St<T>::rnd(v[0]));
    r[(size_t)m * ldr + n] = y;
    rf[frag_index(m, n, ldr >> 5)] = y;
    return St<T>::ld(y);
  }
};

// n < HD: q; else k / v into ring slot pos (fixed, or *pos_ptr) of the caches
// laid out (R, H, Lmax, 64).
template <typename T>
struct BQKV {
  T* q;
  T* kc;
  T* vc;
  int HD, H, Lmax, pos;
  const int* pos_ptr;
  __device__ void operator()(int m, int n, const float (&v)[1]) const {
    const T o = St<T>::st(v[0]);
    const int which = n / HD, nn = n - which * HD;
    if (which == 0) {
      q[(size_t)m * HD + nn] = o;
    } else {
      const int p = pos_ptr ? *pos_ptr : pos;
      T* c = which == 1 ? kc : vc;
      c[(((size_t)m * H + (nn >> 6)) * Lmax + p) * 64 + (nn & 63)] = o;
    }
  }
};

// Rows m = P * pos + r (the positions of one frame, rows r = 0..P-1 each):
// q -> Q row m; k / v -> ring slot pos of ring row r, caches (P, H, Lmax, 64).
template <typename T>
struct BQKVPos {
  T* q;
  T* kc;
  T* vc;
  int HD, H, Lmax, P;
  __device__ void operator()(int m, int n, const float (&v)[1]) const {
    const T o = St<T>::st(v[0]);
    const int which = n / HD, nn = n - which * HD;
    if (which == 0) {
      q[(size_t)m * HD + nn] = o;
    } else {
      const int r = m % P, pos = m / P;
      T* c = which == 1 ? kc : vc;
      c[(((size_t)r * H + (nn >> 6)) * Lmax + pos) * 64 + (nn & 63)] = o;
    }
  }
};

// Output (M, F) in fragment order: the input of the down projection.
template <typename T>
struct BGeglu {
  T* h;
  int F;
  __device__ void operator()(int m, int j, const float (&v)[2]) const {
    const float g = gelu_t<T>(St<T>::rnd(v[0]));
    h[frag_index(m, j, F >> 5)] = St<T>::st(g * St<T>::rnd(v[1]));
  }
};

__device__ __forceinline__ int bg_geglu_row(int j, int p) { return (j >> 5) * 64 + (j & 31) + 32 * p; }

// An input that is normalised (BNorm): the norm weights, and the row sums of
// squares as `parts` partials per row at ssq + m * parts, summed in order.
template <typename T>
struct BNormDev {
  const T* g;
  const float* ssq;
  int parts;
  float eps;
};

// Sum over each 16-lane row of a wave, complete in the row's last lane.
__device__ __forceinline__ float row16_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));   // quad [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));   // quad [2,3,0,1]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));  // row_shr:4
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, true));  // row_shr:8
  return v;
}

// Sum over each 8 lanes, in every lane: pairs, quads, then the other quad.
__device__ __forceinline__ float group8_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));   // quad [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));   // quad [2,3,0,1]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));  // row_half_mirror
  return v;
}

// Eight activations x normalised as rmsnorm_rows rounds them: x times the row's
// inverse RMS, rounded, times the norm weights, rounded.
template <typename T>
__device__ __forceinline__ uint4 norm8(uint4 x, uint4 g, float inv) {
  using S = St<T>;
  const T* xe = reinterpret_cast<const T*>(&x);
  const T* ge = reinterpret_cast<const T*>(&g);
  uint4 out;
  T* oe = reinterpret_cast<T*>(&out);
#pragma unroll
  for (int e = 0; e < 8; ++e) oe[e] = S::st(S::rnd(S::ld(xe[e]) * inv) * S::ld(ge[e]));
  return out;
}

template <class Epi, class = void>
struct HasPre {
  static constexpr bool value = false;
};
template <class Epi>
struct HasPre<Epi, decltype((void)Epi::kPre)> {
  static constexpr bool value = Epi::kPre;
};

template <class Epi>
struct IsResid : std::false_type {};
template <typename T>
struct IsResid<BResid<T>> : std::true_type {};

// Y (M x nout) = X (M x K) . W^T with epilogue, X and W in fragment order.
// P = 1: output n is weight row w_row0 + n; P = 2: output j meets the gate / up
// rows of the packed wi_0 / wi_1 matrix.  Operand fragments of the 16x16x32
// MFMA: lane l holds row (l % 16) of A and column (l % 16) of B over
// k = 8 (l / 16) .. + 7 of the step; the 4 accumulators of lane l hold column
// l % 16, rows 4 (l / 16) + i.  Wave w of the 8 takes k-steps w, w + 8, ...; the
// 8 partial tiles are summed in wave order.  Rows past M repeat the last row and
// columns past nout meet other rows' weights; neither is stored.
//
// NORM: X holds raw residual rows, and a wave normalises its operands between
// their load and the products, rounded as the separate norm rounds them
// (modules.cpp:72-84): a norm folded into the weights would round those once more,
// and below the smallest normal fp16 value lose their bits.  The row's inverse RMS
// (partials, square root, a barrier) and the normalised operands are computed while
// the weights are in flight: those are requested last, as loads return in order
// (32 streams x 50 frames 183.5 ms; weights first 190.2).
//
// Block (tile, ms) of the grid computes output columns [16 C tile, +16 C) for the
// MT row tiles [MT ms, +MT) of 16 rows: blocks sharing a column tile are
// tile + ntiles * ms, on the same XCD as ntiles is then padded to a multiple of
// 8 (blocks are dealt to the 8 XCDs in turn), so the weight tile comes from HBM
// once and from that XCD's L2 for the others.
//
// What bounds it is the launch and one or two memory round trips, so a wave
// requests the operands of NST of its k-steps at once, without a branch between
// the loads (a step past the end re-reads the last one and is not multiplied).
// Fragment order is what makes that pay: rows 2 KB apart put the 16 rows of an
// operand load into few L2 channels, and more of them in flight ran slower
// (64 rows, alone, us: 3,072 outputs 6.6 row-major, 4.1 here; 2,816 gated pairs
// 9.2, 5.8; 1,024 outputs 3.9, 2.9 at K = 1,024 and 6.8, 4.2 at K = 2,816; an
// empty launch takes 1.9; inputs that are not normalised.  In a traced frame, with
// normalised inputs: 6.8, 9.8 and 4.8; residual outputs 3.9 and 4.8).
template <typename T, int P, int C, int MT, int NST, bool NORM, class Epi>
__global__ __launch_bounds__(kBgThreads) void k_bgemm(const T* __restrict__ X, int M, int K, const T* __restrict__ W,
                                                      int nout, int ntiles, Epi epi, int w_row0, int w_group_rows,
                                                      BNormDev<T> nrm) {
  static_assert(P == 1 || C == 1, "gate / up pairs: one column tile a block");
  static_assert(C == 1 || !HasPre<Epi>::value, "the residual epilogue: one column tile a block");
  // blockIdx.y = group g (grouped launch): rows [g M, g M + M) of X against
  // weight rows w_row0 + g * w_group_rows, outputs at rows g M + m
  const int grow = blockIdx.y * M;
  const int row0 = w_row0 + blockIdx.y * w_group_rows, skip = P == 1 ? row0 & 15 : 0;
  constexpr int kW = P * C;                                    // weight tiles of the block
  constexpr int kRows = 16 * MT;
  constexpr int kOut = kRows * kBgCols;                        // outputs of a column tile
  constexpr int kPer = (kOut + kBgThreads - 1) / kBgThreads;  // of them per thread
  __shared__ float part[kBgWaves][kRows][kBgCols + 1];  // one weight tile at a time
  [[maybe_unused]] __shared__ float inv_s[kRows];
  // the wave index as a scalar: matrix instructions ignore the lane mask, so the
  // conditions around them must be branches
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = (blockIdx.x % ntiles) * C, m0 = (blockIdx.x / ntiles) * kRows;
  const int j0 = tile * kBgCols - skip;  // output of the block's first column
  if (j0 >= nout) return;                // a padding tile (launch_bgemm_t)
  const int c16 = lane & 15, kg = lane >> 4;
  const int nks = K / 32;

  // weight tile w of k-step ks: the P parts of an output tile alternate, column
  // tiles lie a whole K apart
  const T* wt = W + ((size_t)(P == 1 ? (row0 >> 4) + tile : tile) * nks * P) * 512 + lane * 8;
  const T* xrow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int r = grow + min(m0 + 16 * t + c16, M - 1);
    xrow[t] = X + (size_t)(r >> 4) * nks * 512 + (kg * 16 + (r & 15)) * 8;
  }
  uint4 b[NST][kW], a[NST][MT];
  [[maybe_unused]] uint4 gk[NORM ? NST : 1];
  auto weights = [&](int c, int ks) {
#pragma unroll
    for (int w = 0; w < kW; ++w) b[c][w] = ld_g16(wt + (size_t)(C == 1 ? ks * P + w : w * nks + ks) * 512);
  };
  auto load = [&](int s0) {
#pragma unroll
    for (int c = 0; c < NST; ++c) {
      const int ks = min(s0 + kBgWaves * c, nks - 1);
#pragma unroll
      for (int t = 0; t < MT; ++t) a[c][t] = ld_g16(xrow[t] + (size_t)ks * 512);
      if constexpr (NORM) gk[c] = ld_g16(nrm.g + ks * 32 + kg * 8);
      if constexpr (!NORM) weights(c, ks);
    }
    if constexpr (NORM) {  // the weights last: the rest is at work before they are there
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < NST; ++c) weights(c, min(s0 + kBgWaves * c, nks - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // eight lanes per row r: with 64 partials lane q sums [8 q, 8 q + 8) in order
  // (other counts: lane 0 sums them all)
  [[maybe_unused]] const int r = tid >> 3, q = tid & 7;
  [[maybe_unused]] float4 su, sw;
  [[maybe_unused]] const float* sp = nullptr;
  if constexpr (NORM) {
    sp = nrm.ssq + (size_t)(grow + min(m0 + min(r, kRows - 1), M - 1)) * nrm.parts;
    if (nrm.parts == 64) {
      su = *reinterpret_cast<const float4*>(sp + 8 * q);
      sw = *reinterpret_cast<const float4*>(sp + 8 * q + 4);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  load(wid);
  float pre[kPer];
  if constexpr (HasPre<Epi>::value) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int idx = min(tid + kBgThreads * i, kOut - 1), m = m0 + idx / kBgCols, n = j0 + idx % kBgCols;
      pre[i] = epi.pre(grow + min(m, M - 1), min(n, nout - 1));
    }
  }
  [[maybe_unused]] float inv[MT];
  if constexpr (NORM) {
    float ss = 0.f;
    if (nrm.parts == 64) {
      ss = ((((((su.x + su.y) + su.z) + su.w) + sw.x) + sw.y) + sw.z) + sw.w;
    } else if (q == 0) {
      for (int t = 0; t < nrm.parts; ++t) ss += sp[t];
    }
    ss = group8_sum(ss);
    if (r < kRows && q == 0) inv_s[r] = 1.0f / sqrtf(ss / (float)K + nrm.eps);
    ring_barrier();  // not __syncthreads(): the operands stay in flight
#pragma unroll
    for (int t = 0; t < MT; ++t) inv[t] = inv_s[16 * t + c16];
  }
  f32x4_t acc[kW][MT];
#pragma unroll
  for (int w = 0; w < kW; ++w)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[w][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  for (int s0 = wid; s0 < nks; s0 += kBgWaves * NST) {
    if constexpr (NORM) {
#pragma unroll
      for (int c = 0; c < NST; ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t) a[c][t] = norm8<T>(a[c][t], gk[c], inv[t]);
    }
#pragma unroll
    for (int c = 0; c < NST; ++c) {
      if (s0 + kBgWaves * c < nks) {
#pragma unroll
        for (int w = 0; w < kW; ++w)
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[w][t] = Mfma16<T>::mma(a[c][t], b[c][w], acc[w][t]);
      }
    }
    if (s0 + kBgWaves * NST < nks) load(s0 + kBgWaves * NST);
  }
#pragma unroll
  for (int ct = 0; ct < C; ++ct) {
    float v[kPer][P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      if (ct + p > 0) __syncthreads();  // the previous weight tile's sums have been read
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wid][16 * t + 4 * kg + i][c16] = acc[ct + p][t][i];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int idx = min(tid + kBgThreads * i, kOut - 1), m = idx / kBgCols, n = idx % kBgCols;
        float sum = part[0][m][n];
#pragma unroll
        for (int w = 1; w < kBgWaves; ++w) sum += part[w][m][n];
        v[i][p] = sum;
      }
    }
    if constexpr (IsResid<Epi>::value) {
      // lanes 16 r .. 16 r + 15 of a wave hold the 16 columns of one output row
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int idx = tid + kBgThreads * i, m = m0 + idx / kBgCols, n = idx % kBgCols;
        const bool ok = idx < kOut && m < M && j0 + n < nout;
        const float y = ok ? epi(grow + m, j0 + n, v[i], pre[i]) : 0.f;
        const float ss = row16_sum(y * y);
        if (ok && n == kBgCols - 1) epi.ssq[(size_t)(grow + m) * (epi.ldr / kBgCols) + tile] = ss;
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int idx = tid + kBgThreads * i, m = m0 + idx / kBgCols, n = j0 + ct * kBgCols + idx % kBgCols;
        if (idx >= kOut || m >= M || n < 0 || n >= nout) continue;
        epi(grow + m, n, v[i]);
      }
    }
  }
}

// Row tiles per block: grids of fewer than 128 column tiles (the d_model-wide
// outputs) split the rows until there are 256 blocks, one per CU; wider
// outputs keep all rows in a block (each block then reads the activations once
// for twice the columns' work), the gated pairs at most two row tiles (64 rows:
// 5.8 against 6.5 us with four).  Where the input is normalised, a block of the
// wide outputs takes two column tiles and two row tiles instead of one and four:
// as many products, half the rows to normalise.  A block holds 1, 2 or 4 row tiles, no more
// than the rows need: the loads of unused ones cost as much (the 3,072-wide
// output of 10 rows: 8.5 us with four).
template <typename T, int P, bool NORM, class Epi>
void launch_bgemm_t(const T* X, int M, int K, const T* W, int nout, const Epi& epi, hipStream_t s, int groups,
                    int w_row0, int w_group_rows, const BNormDev<T>& nrm) {
  // a column tile more where the weight rows do not start on a tile
  const bool shifted = P == 1 && (w_row0 % kBgCols != 0 || (groups > 1 && w_group_rows % kBgCols != 0));
  const int ntiles = (nout + kBgCols - 1) / kBgCols + (shifted ? 1 : 0), mtiles = (M + 15) / 16;
  int ms = 1;
  while (ntiles < 128 && ms < 4 && ms < mtiles && ntiles * ms < 256) ms *= 2;
  const int mt = (mtiles + ms - 1) / ms;
  auto go = [&](auto k, int mt_block, int c_block = 1) {
    const int mb = (mtiles + mt_block - 1) / mt_block, nb = (ntiles + c_block - 1) / c_block;
    const int nt = mb > 1 ? (nb + 7) / 8 * 8 : nb;
    hipLaunchKernelGGL(k, dim3(nt * mb, groups), dim3(kBgThreads), 0, s, X, M, K, W, nout, nt, epi, w_row0,
                       w_group_rows, nrm);
  };
  // 12 steps in flight cover K <= 3072 with one row tile
  if (mt == 1 && P == 1 && K > 32 * 4 * kBgWaves)
    go(k_bgemm<T, P, 1, 1, P == 1 ? 12 : 4, NORM, Epi>, 1);
  else if (mt == 1)
    go(k_bgemm<T, P, 1, 1, 4, NORM, Epi>, 1);
  else if (mt == 2 || P == 2)
    go(k_bgemm<T, P, 1, 2, 4, NORM, Epi>, 2);
  else if (NORM && !shifted && nout % (2 * kBgCols) == 0)
    go(k_bgemm<T, P, NORM && P == 1 && !HasPre<Epi>::value ? 2 : 1, 2, 4, NORM, Epi>, 2, 2);
  else
    go(k_bgemm<T, P, 1, P == 2 ? 2 : 4, 4, NORM, Epi>, 4);
  MRT_HIP_CHECK(hipGetLastError());
}

template <typename T, int P, class Epi>
void launch_bgemm(const void* X, int M, int K, const void* W, int nout, const Epi& epi, hipStream_t s,
                  const BNorm& norm = {}, int w_row0 = 0, int groups = 1, int w_group_rows = 0) {
  MRT_REQUIRE(M >= 1 && M * groups <= kBatchRows, "batched GEMM: rows must be in [1, 64]");
  MRT_REQUIRE(K % 32 == 0 && K >= 32, "batched GEMM: K must be a multiple of 32");
  MRT_REQUIRE(nout >= 1 && groups >= 1 && w_row0 >= 0, "batched GEMM: no outputs");
  const T* x = static_cast<const T*>(X);
  const T* w = static_cast<const T*>(W);
  if constexpr (!HasPre<Epi>::value) {  // the residual update's input is never normalised
    if (norm.g != nullptr) {
      MRT_REQUIRE(norm.ssq != nullptr, "batched GEMM: a normalised input needs its row partials");
      launch_bgemm_t<T, P, true>(x, M, K, w, nout, epi, s, groups, w_row0, w_group_rows,
                                 BNormDev<T>{static_cast<const T*>(norm.g), norm.ssq, K / kBgCols, norm.eps});
      return;
    }
  }
  launch_bgemm_t<T, P, false>(x, M, K, w, nout, epi, s, groups, w_row0, w_group_rows,
                              BNormDev<T>{nullptr, nullptr, 0, 0.f});
}

// The same product with every output's sum taken over k in order in one accumulator,
// as the encoder's GEMM takes it (a chain of 16x16x32 instructions gives bit for bit
// what its 32x32x16 chain gives), for the full-sequence depth pass: its logits do not
// depend on which GEMM ran.  A block is one wave: NW weight tiles (the P parts of an
// output tile, or column tiles) against one row tile.  The chain is short (0.5 us at
// K = 1,024); what bounds it is the operands' round trip, so a wave keeps two runs of
// kSeqRun k-steps requested, all of K = 1,024.
constexpr int kSeqRun = 16;

template <typename T>
struct SResid {
  T* r;
  int ldr;
  static constexpr bool kPre = true;
  __device__ float pre(int m, int n) const { return St<T>::ld(r[(size_t)m * ldr + n]); }
  __device__ void operator()(int m, int n, const float (&v)[1], float x) const {
    r[(size_t)m * ldr + n] = St<T>::st(x + St<T>::rnd(v[0]));
  }
};

template <typename T, int P, int NW, class Epi>
__global__ __launch_bounds__(64) void k_bgemm_seq(const T* __restrict__ X, int M, int K, const T* __restrict__ W,
                                                  int nout, Epi epi) {
  static_assert(P == 1 || NW == P, "gate / up pairs: one column tile a block");
  constexpr int C = NW / P;
  const int lane = threadIdx.x, c16 = lane & 15, kg = lane >> 4, nks = K / 32;
  // eight columns of blocks, then the same eight for the next row tile: blocks of one
  // column run together on one XCD (blocks are dealt to the 8 XCDs in turn)
  const int mt = (M + 15) / 16, id = blockIdx.x / 8;
  const int tile = (id / mt * 8 + blockIdx.x % 8) * C, m0 = id % mt * 16;
  if (tile * kBgCols >= nout) return;
  const T* wt = W + (size_t)tile * nks * P * 512 + lane * 8;
  const int r = min(m0 + c16, M - 1);
  const T* xr = X + (size_t)(r >> 4) * nks * 512 + (kg * 16 + (r & 15)) * 8;
  float pre[C][4];
  if constexpr (HasPre<Epi>::value) {
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        pre[c][i] = epi.pre(min(m0 + 4 * kg + i, M - 1), min((tile + c) * kBgCols + c16, nout - 1));
  }
  uint4 a[2][kSeqRun], b[2][kSeqRun][NW];
  auto load = [&](int d, int s0) {  // a step past the end re-reads the last one and is not multiplied
#pragma unroll
    for (int s = 0; s < kSeqRun; ++s) {
      const int ks = min(s0 + s, nks - 1);
#pragma unroll
      for (int w = 0; w < NW; ++w) b[d][s][w] = ld_g16(wt + (size_t)(P == 1 ? w * nks + ks : ks * P + w) * 512);
      a[d][s] = ld_g16(xr + (size_t)ks * 512);
    }
  };
  f32x4_t acc[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w) acc[w] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto run = [&](int d, int s0) {
#pragma unroll
    for (int s = 0; s < kSeqRun; ++s)
      if (s0 + s < nks) {  // uniform: a branch, matrix instructions ignore the lane mask
#pragma unroll
        for (int w = 0; w < NW; ++w) acc[w] = Mfma16<T>::mma(a[d][s], b[d][s][w], acc[w]);
      }
    if (s0 + 2 * kSeqRun < nks) load(d, s0 + 2 * kSeqRun);
  };
  load(0, 0);
  if (kSeqRun < nks) load(1, kSeqRun);
  for (int s0 = 0; s0 < nks; s0 += 2 * kSeqRun) {
    run(0, s0);
    if (s0 + kSeqRun < nks) run(1, s0 + kSeqRun);
  }
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + 4 * kg + i, n = (tile + c) * kBgCols + c16;
      if (m >= M || n >= nout) continue;
      float v[P];
#pragma unroll
      for (int p = 0; p < P; ++p) v[p] = acc[c * P + p][i];
      if constexpr (HasPre<Epi>::value)
        epi(m, n, v, pre[c][i]);
      else
        epi(m, n, v);
    }
}

// Two column tiles a wave where that still leaves several waves a CU (the head): half
// the reads of X.
template <typename T, int P, class Epi>
void launch_bgemm_seq(const void* X, int M, int K, const void* W, int nout, const Epi& epi, hipStream_t s) {
  MRT_REQUIRE(M >= 1 && K % 32 == 0 && K >= 32 && nout >= 1, "sequential GEMM: K must be a multiple of 32");
  const int tiles = (nout + kBgCols - 1) / kBgCols, mt = (M + 15) / 16;
  const T *x = static_cast<const T*>(X), *w = static_cast<const T*>(W);
  if (P == 1 && tiles * mt >= 1024)
    hipLaunchKernelGGL((k_bgemm_seq<T, P, 2, Epi>), dim3((tiles + 15) / 16 * 8 * mt), dim3(64), 0, s, x, M, K, w, nout, epi);
  else
    hipLaunchKernelGGL((k_bgemm_seq<T, P, P, Epi>), dim3((tiles + 7) / 8 * 8 * mt), dim3(64), 0, s, x, M, K, w, nout, epi);
  MRT_HIP_CHECK(hipGetLastError());
}

// Weights (N, K) -> fragment order.  Block (tile, ks): 16 rows x 32 columns a
// part; P = 2: the gate and up rows of 16 outputs of a packed matrix.  Rows past
// N are zero.
template <typename T, int P>
__global__ __launch_bounds__(64) void k_frag_weights(const T* __restrict__ W, int N, int K, T* __restrict__ out) {
  const int tile = blockIdx.x, ks = blockIdx.y, lane = threadIdx.x, nks = K / 32;
  const int k0 = ks * 32 + (lane >> 4) * 8;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int j = tile * 16 + (lane & 15), row = P == 1 ? j : bg_geglu_row(j, p);
    const uint4 v = row < N ? ld_g16(W + (size_t)row * K + k0) : make_uint4(0u, 0u, 0u, 0u);
    *reinterpret_cast<uint4*>(out + (((size_t)tile * nks + ks) * P + p) * 512 + lane * 8) = v;
  }
}

// Cross attention of one (row, head) over all S encoder keys (no bias, no
// mask, scale 1.0: modules.cpp:243-295), one 256-thread block per pair.  A
// wave reads 8 whole K (then V) rows per 16-byte load instruction: thread t
// owns the 8-dim slice t % 8 of keys t / 8, t / 8 + 32, ...; scores are
// reduced over the 8 slices with lane shuffles and kept in LDS; the softmax
// weights then scale V the same way and the 32 key groups are summed in a
// fixed order.
constexpr int kCrossMaxS = 1024;

__global__ __launch_bounds__(256) void k_cross_attn_b(const bf16* __restrict__ Q, const bf16* __restrict__ Kc,
                                                      const bf16* __restrict__ Vc, int H, int S, bf16* __restrict__ out) {
  __shared__ float qs[64];
  __shared__ float ps[kCrossMaxS];
  __shared__ float red[32][65];
  __shared__ float wred[2][4];
  const int bh = blockIdx.x, b = bh / H, h = bh - b * H;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int d8 = tid & 7, kg = tid >> 3;
  const int HD = H * 64;
  if (tid < 64) qs[tid] = St<bf16>::ld(Q[(size_t)b * HD + h * 64 + tid]);
  __syncthreads();
  float q[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e] = qs[8 * d8 + e];
  const bf16* Kp = Kc + (size_t)bh * S * 64 + 8 * d8;
  const bf16* Vp = Vc + (size_t)bh * S * 64 + 8 * d8;
  float mx = -INFINITY;
  for (int j0 = 0; j0 < S; j0 += 4 * 32) {
    uint4 kv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + kg + 32 * u;
      kv[u] = j < S ? ld_nt16(Kp + (size_t)j * 64) : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bf16* ke = reinterpret_cast<const bf16*>(&kv[u]);
      float sc = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) sc = fmaf(q[e], St<bf16>::ld(ke[e]), sc);
      sc += __shfl_xor(sc, 1, 64);
      sc += __shfl_xor(sc, 2, 64);
      sc += __shfl_xor(sc, 4, 64);
      const int j = j0 + kg + 32 * u;
      if (j < S) {
        if (d8 == 0) ps[j] = sc;
        mx = fmaxf(mx, sc);
      }
    }
  }
  mx = wave_max(mx);
  if (lane == 0) wred[0][wid] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(wred[0][0], wred[0][1]), fmaxf(wred[0][2], wred[0][3]));
  float sum = 0.f;
  for (int j = tid; j < S; j += 256) {
    const float e = expf(ps[j] - mx);
    ps[j] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) wred[1][wid] = sum;
  __syncthreads();
  sum = (wred[1][0] + wred[1][1]) + (wred[1][2] + wred[1][3]);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < S; j0 += 4 * 32) {
    uint4 vv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + kg + 32 * u;
      vv[u] = j < S ? ld_nt16(Vp + (size_t)j * 64) : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + kg + 32 * u;
      const float pj = j < S ? ps[j] : 0.f;
      const bf16* ve = reinterpret_cast<const bf16*>(&vv[u]);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(pj, St<bf16>::ld(ve[e]), acc[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[kg][8 * d8 + e] = acc[e];
  __syncthreads();
  if (tid < 64) {
    float o = 0.f;
    for (int g = 0; g < 32; ++g) o += red[g][tid];
    out[frag_index(b, h * 64 + tid, HD >> 5)] = St<bf16>::st(o / sum);
  }
}

// Gumbel noise of every draw of a chunk for every stream: out (B, frames, L, C)
// = gumbel(seeds[b], frame, level, i), the values the sampler would compute.
__global__ void k_gumbel_tables(const uint64_t* __restrict__ seeds, int frames, int L, int C, int n,
                                float* __restrict__ out) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = i % C, r = i / C, level = r % L, r2 = r / L, frame = r2 % frames, b = r2 / frames;
    out[i] = gumbel(seeds[b], frame, level, c);
  }
}

__global__ void k_set_counter(int* p, int v) { *p = v; }
__global__ void k_advance_counter(int* p) { *p = *p + 1; }

}  // namespace

void gumbel_tables(const uint64_t* seeds, int streams, int frames, int L, int C, float* out, hipStream_t s) {
  const long n = (long)streams * frames * L * C;
  MRT_REQUIRE(n > 0 && n < (1L << 31), "gumbel tables: size out of range");
  const int blocks = (int)std::min<long>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_gumbel_tables, dim3(blocks), dim3(256), 0, s, seeds, frames, L, C, (int)n, out);
  MRT_HIP_CHECK(hipGetLastError());
}

void set_counter(int* p, int v, hipStream_t s) {
  hipLaunchKernelGGL(k_set_counter, dim3(1), dim3(1), 0, s, p, v);
  MRT_HIP_CHECK(hipGetLastError());
}

void advance_counter(int* p, hipStream_t s) {
  hipLaunchKernelGGL(k_advance_counter, dim3(1), dim3(1), 0, s, p);
  MRT_HIP_CHECK(hipGetLastError());
}

void cross_attn_rows(const void* Q, const void* Kc, const void* Vc, int rows, int H, int S, void* out, hipStream_t s) {
  MRT_REQUIRE(S >= 1 && S <= kCrossMaxS, "batched cross attention: encoder length must be in [1, 1024]");
  hipLaunchKernelGGL(k_cross_attn_b, dim3(rows * H), dim3(256), 0, s, static_cast<const bf16*>(Q),
                     static_cast<const bf16*>(Kc), static_cast<const bf16*>(Vc), H, S, static_cast<bf16*>(out));
  MRT_HIP_CHECK(hipGetLastError());
}

#define MRT_DTYPE16(dt, ...)                                                         \
  do {                                                                               \
    MRT_REQUIRE((dt) != DType::F32, "batched GEMM: 16-bit storage types only");      \
    if ((dt) == DType::BF16) {                                                       \
      using T = bf16;                                                                \
      __VA_ARGS__;                                                                   \
    } else {                                                                         \
      using T = f16;                                                                 \
      __VA_ARGS__;                                                                   \
    }                                                                                \
  } while (0)

// One tile more than the rows fill: a range of weight rows that does not start
// on a tile may touch it (its outputs are not stored).
size_t frag_weights_elems(int N, int K) { return (static_cast<size_t>((N + 15) / 16) + 1) * 16 * K; }

void frag_weights(DType dt, const void* W, int N, int K, bool pairs, void* out, hipStream_t s) {
  MRT_REQUIRE(K % 32 == 0 && N >= 1, "fragment weights: K must be a multiple of 32");
  MRT_REQUIRE(!pairs || N % 64 == 0, "fragment weights: gate / up pairs come in groups of 64 rows");
  const int tiles = (pairs ? N / 2 : N + 15) / 16;
  MRT_DTYPE16(dt, {
    const auto k = pairs ? k_frag_weights<T, 2> : k_frag_weights<T, 1>;
    hipLaunchKernelGGL(k, dim3(tiles, K / 32), dim3(64), 0, s, static_cast<const T*>(W), N, K,
                       static_cast<T*>(out));
  });
  MRT_HIP_CHECK(hipGetLastError());
}

void bgemm_store(DType dt, const void* X, int M, int K, const void* W, int N, void* Y, int ldy, hipStream_t s,
                 const BNorm& norm) {
  MRT_DTYPE16(dt, (launch_bgemm<T, 1>(X, M, K, W, N, BStore<T>{static_cast<T*>(Y), ldy}, s, norm)));
}

void bgemm_f32(DType dt, const void* X, int M, int K, const void* W, int w_row0, int N, float* Y, int ldy,
               hipStream_t s, const BNorm& norm, int groups, int w_group_rows) {
  MRT_DTYPE16(dt, (launch_bgemm<T, 1>(X, M, K, W, N, BF32<T>{Y, ldy}, s, norm, w_row0, groups, w_group_rows)));
}

void bgemm_resid(DType dt, const void* X, int M, int K, const void* W, int N, void* R, void* Rf, float* ssq,
                 hipStream_t s) {
  MRT_REQUIRE(N % 32 == 0, "batched GEMM: residual rows must be whole fragments");
  MRT_DTYPE16(dt, (launch_bgemm<T, 1>(X, M, K, W, N, BResid<T>{static_cast<T*>(R), N, static_cast<T*>(Rf), ssq}, s)));
}

void bgemm_qkv(DType dt, const void* X, int M, int K, const void* W, int HD, void* Q, void* Kc, void* Vc, int H,
               int Lmax, int pos, const int* pos_ptr, hipStream_t s, const BNorm& norm) {
  MRT_DTYPE16(dt, (launch_bgemm<T, 1>(X, M, K, W, 3 * HD,
                                      BQKV<T>{static_cast<T*>(Q), static_cast<T*>(Kc), static_cast<T*>(Vc), HD, H,
                                              Lmax, pos, pos_ptr},
                                      s, norm)));
}

void bgemm_qkv_pos(DType dt, const void* X, int M, int K, const void* W, int HD, void* Q, void* Kc, void* Vc, int H,
                   int Lmax, int P, hipStream_t s) {
  MRT_REQUIRE(P >= 1 && M % P == 0 && M / P <= Lmax, "batched GEMM: positions exceed the ring");
  MRT_DTYPE16(dt, (launch_bgemm<T, 1>(X, M, K, W, 3 * HD,
                                      BQKVPos<T>{static_cast<T*>(Q), static_cast<T*>(Kc), static_cast<T*>(Vc), HD, H,
                                                 Lmax, P},
                                      s)));
}

void bgemm_geglu(DType dt, const void* X, int M, int K, const void* W01, int F, void* Hout, hipStream_t s,
                 const BNorm& norm) {
  MRT_REQUIRE(F % 32 == 0, "batched GEMM: d_ff must be a multiple of 32 (packed gate/up groups)");
  MRT_DTYPE16(dt, (launch_bgemm<T, 2>(X, M, K, W01, F, BGeglu<T>{static_cast<T*>(Hout), F}, s, norm)));
}

void bgemm_seq_store(DType dt, const void* X, int M, int K, const void* W, int N, void* Y, hipStream_t s) {
  MRT_DTYPE16(dt, (launch_bgemm_seq<T, 1>(X, M, K, W, N, BStore<T>{static_cast<T*>(Y), N}, s)));
}

void bgemm_seq_f32(DType dt, const void* X, int M, int K, const void* W, int N, float* Y, hipStream_t s) {
  MRT_DTYPE16(dt, (launch_bgemm_seq<T, 1>(X, M, K, W, N, BF32<T>{Y, N}, s)));
}

void bgemm_seq_resid(DType dt, const void* X, int M, int K, const void* W, int N, void* R, hipStream_t s) {
  MRT_DTYPE16(dt, (launch_bgemm_seq<T, 1>(X, M, K, W, N, SResid<T>{static_cast<T*>(R), N}, s)));
}

void bgemm_seq_geglu(DType dt, const void* X, int M, int K, const void* W01, int F, void* Hout, hipStream_t s) {
  MRT_REQUIRE(F % 32 == 0, "sequential GEMM: d_ff must be a multiple of 32 (packed gate/up groups)");
  MRT_DTYPE16(dt, (launch_bgemm_seq<T, 2>(X, M, K, W01, F, BGeglu<T>{static_cast<T*>(Hout), F}, s)));
}

}  // namespace mrt
