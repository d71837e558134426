// Once-per-chunk encoder prefill kernels for gfx950 (model.cpp:226-241,
// modules.cpp:339-358) and the cross-attention K/V projection of every
// temporal layer (modules.cpp:448-455) as one wide GEMM.
//
// GEMM operands are both K-contiguous ("NT": activations (M, K) row-major,
// weights (N, K) row-major as the bundle stores them).  bf16 and fp16 use
// v_mfma_f32_32x32x16_{bf16,f16} through the LDS ring of ring_gemm.hpp; fp32 splits its
// operands into three bf16 parts for the same instruction (split_gemm.hpp), or
// uses a VALU tile where the shapes do not fit.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device_utils.hpp"
#include "kernels.hpp"
#include "mfma_ring.hpp"
#include "split_gemm.hpp"

namespace mrt {
namespace {

// ---- embedding + position embedding ------------------------------------------
template <typename T>
__global__ void k_encoder_embed(const T* __restrict__ emb, const T* __restrict__ pe,
                                const int* __restrict__ tok, int S, int D, T* __restrict__ x) {
  const int r = blockIdx.x, s = r % S;
  const T* e = emb + (size_t)tok[r] * D;
  const T* p = pe + (size_t)s * D;
  for (int d = threadIdx.x; d < D; d += blockDim.x)
    x[(size_t)r * D + d] = St<T>::st(St<T>::ld(e[d]) + St<T>::ld(p[d]));
}

// Where a norm leaves element d of row r: row-major, or in the fragment order of the
// skinny GEMMs (batch.hpp; D % 32 == 0).
template <bool FRAG>
__device__ __forceinline__ size_t norm_index(int r, int d, int D) {
  return FRAG ? frag_index(r, d, D >> 5) : (size_t)r * D + d;
}

// Rows of up to 256 * kNormPer elements: each thread keeps its elements in
// registers between the sum of squares and the scaling (one read of x).
constexpr int kNormPer = 8;

template <typename T, bool FRAG>
__global__ __launch_bounds__(256) void k_rmsnorm_rows_reg(const T* __restrict__ x, const T* __restrict__ g,
                                                          float eps, int D, T* __restrict__ y) {
  using S = St<T>;
  __shared__ float red[4];
  const int r = blockIdx.x, tid = threadIdx.x;
  const T* xr = x + (size_t)r * D;
  float v[kNormPer];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kNormPer; ++i) {
    const int d = tid + 256 * i;
    v[i] = d < D ? S::ld(xr[d]) : 0.f;
    ss += v[i] * v[i];
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)D + eps);
#pragma unroll
  for (int i = 0; i < kNormPer; ++i) {
    const int d = tid + 256 * i;
    if (d < D) y[norm_index<FRAG>(r, d, D)] = S::st(S::rnd(v[i] * inv) * S::ld(g[d]));
  }
}

// One wave per row of D = 64 V NV elements (V per 16-byte chunk): a lane keeps
// its NV chunks in registers between the sum of squares and the scaling, and
// the row's sum is one wave reduction (no LDS, no barrier); four rows per block.
template <typename T, int NV, bool FRAG>
__global__ __launch_bounds__(256) void k_rmsnorm_rows_wave(const T* __restrict__ x, const T* __restrict__ g,
                                                           float eps, int M, int D, T* __restrict__ y) {
  using S = St<T>;
  constexpr int V = S::kVec;
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);  // wave-uniform
  if (r >= M) return;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (size_t)r * D);
  const uint4* gr = reinterpret_cast<const uint4*>(g);
  uint4 v[NV], gv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = xr[lane + 64 * i];
#pragma unroll
  for (int i = 0; i < NV; ++i) gv[i] = gr[lane + 64 * i];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const T* e = reinterpret_cast<const T*>(&v[i]);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const float f = S::ld(e[k]);
      ss += f * f;
    }
  }
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const T* e = reinterpret_cast<const T*>(&v[i]);
    const T* ge = reinterpret_cast<const T*>(&gv[i]);
    uint4 o;
    T* oe = reinterpret_cast<T*>(&o);
#pragma unroll
    for (int k = 0; k < V; ++k) oe[k] = S::st(S::rnd(S::ld(e[k]) * inv) * S::ld(ge[k]));
    *reinterpret_cast<uint4*>(y + norm_index<FRAG>(r, (lane + 64 * i) * V, D)) = o;
  }
}

template <typename T, bool FRAG>
__global__ __launch_bounds__(256) void k_rmsnorm_rows(const T* __restrict__ x, const T* __restrict__ g,
                                                      float eps, int D, T* __restrict__ y) {
  using S = St<T>;
  __shared__ float red[4];
  const int r = blockIdx.x, tid = threadIdx.x;
  const T* xr = x + (size_t)r * D;
  float ss = 0.f;
  for (int d = tid; d < D; d += 256) {
    const float v = S::ld(xr[d]);
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)D + eps);
  for (int d = tid; d < D; d += 256)
    y[norm_index<FRAG>(r, d, D)] = S::st(S::rnd(S::ld(xr[d]) * inv) * S::ld(g[d]));
}

// ---- GEMM epilogue ----------------------------------------------------------------
template <typename T>
struct GemmOut {
  GemmEpiArgs a;
  int N;
  __device__ __forceinline__ void put(int m, int n, float acc) const {
    using S = St<T>;
    T* C = static_cast<T*>(a.C);
    if (a.kind == GemmEpi::Store) {
      C[(size_t)m * N + n] = S::st(acc);
    } else if (a.kind == GemmEpi::Resid) {
      T* p = C + (size_t)m * N + n;
      *p = S::st(S::ld(*p) + S::rnd(acc));
    } else if (a.kind == GemmEpi::StoreF32) {
      static_cast<float*>(a.C)[(size_t)m * N + n] = S::rnd(acc);
    } else {  // CrossKV
      const int lk = n / a.HD, nn = n - lk * a.HD;
      const int h = nn >> 6, d = nn & 63;
      const int b = m / a.S, s = m - b * a.S;
      C[((((size_t)lk * a.nb + b) * a.H + h) * a.S + s) * 64 + d] = S::st(acc);
    }
  }
  // Gated-GELU pair: packed column n (gate, n % 64 < 32) and n + 32 (up).
  __device__ __forceinline__ void put_geglu(int m, int n, float g, float u) const {
    using S = St<T>;
    T* C = static_cast<T*>(a.C);
    const int j = (n >> 6) * 32 + (n & 31);
    const float gl = gelu_t<T>(S::rnd(g));
    C[(size_t)m * (N / 2) + j] = S::st(gl * S::rnd(u));
  }
};

// ---- VALU tiled GEMM (shapes the matrix-core tiles do not take) ---------------------
// 64x64 tile, BK 16, 256 threads, 4x4 outputs per thread at rows ty+16i and
// columns tx+16j, so columns j and j+2 form a packed gate/up pair.
template <typename T>
__global__ __launch_bounds__(256) void k_gemm_valu(const T* __restrict__ A, const T* __restrict__ B,
                                                   int M, int N, int K, GemmOut<T> out) {
  using S = St<T>;
  __shared__ float As[16][64 + 4];
  __shared__ float Bs[16][64 + 4];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i, r = idx >> 4, c = idx & 15;
      const int gm = m0 + r, gn = n0 + r, gk = k0 + c;
      As[c][r] = (gm < M && gk < K) ? S::ld(A[(size_t)gm * K + gk]) : 0.f;
      Bs[c][r] = (gn < N && gk < K) ? S::ld(B[(size_t)gn * K + gk]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty + 16 * i;
    if (m >= M) continue;
    if (out.a.kind == GemmEpi::Geglu) {
#pragma unroll
      for (int j = 0; j < 2; ++j) out.put_geglu(m, n0 + tx + 16 * j, acc[i][j], acc[i][j + 2]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + tx + 16 * j;
        if (n < N) out.put(m, n, acc[i][j]);
      }
    }
  }
}

// ---- matrix-core GEMM ------------------------------------------------------------------
// gelu_t of 16-bit types with tanh taken as (1 - t) / (1 + t), t = 2^(-2 |x| log2 e):
// within 2e-7 of tanhf, far below the 16-bit rounding of 1 + tanh that is all the
// formula keeps of it (every finite bf16 and fp16 value has gelu_t's result).  tanhf's two polynomial paths made the 181 M gated-GELUs of
// 32 streams a 300 us epilogue.
template <typename T>
__device__ __forceinline__ float gelu16(float x) {
  using S = St<T>;
  const float x2 = S::rnd(x * x);
  float t = S::rnd(S::rnd(0.044715f) * x2);
  t = S::rnd(1.0f + t);
  t = S::rnd(x * t);
  const float inner = S::rnd(S::rnd(0.7978845608028654f) * t);
  const float q = __builtin_amdgcn_exp2f(fabsf(inner) * -2.8853900817779268f);
  const float th = S::rnd(copysignf((1.0f - q) * __builtin_amdgcn_rcpf(1.0f + q), inner));
  t = S::rnd(1.0f + th);
  t = S::rnd(x * t);
  return S::rnd(0.5f * t);
}

// Epilogue of a wave's tile, first row mb, first column nb: a lane holds row
// mb + 32 i + lane % 32 of tile (i, j) and four times four consecutive columns
// (j = 2 p / 2 p + 1: gate / up columns of gated-GELU pair p).  16-bit results swap
// halves between lanes l and l + 32, so that a lane stores 8 consecutive columns,
// 16 bytes.  The kind is resolved once per tile, and the residual epilogue loads
// every residual before it stores anything.
template <typename T, int MI, int NJ>
__device__ __forceinline__ void mfma_epilogue(const GemmOut<T>& out, const f32x16_t (&acc)[MI][NJ], int M, int mb,
                                              int nb) {
  using St_ = St<T>;
  constexpr bool k16 = sizeof(T) == 2;
  constexpr int G = k16 ? 2 : 4, V = k16 ? 8 : 4;  // stores per 32 columns, columns per store
  const int lane = threadIdx.x & 63, lh = lane >> 5;
  const int N = out.N, m0 = mb + (lane & 31);
  T* C = static_cast<T*>(out.a.C);
  // the 16 bytes of group g of four (16 bit: groups 2 g and 2 g + 1 of the lane
  // pair) from f(r), r = 0 .. 15, and their first column in the 32
  auto pack = [&](int g, auto&& f) -> uint4 {
    uint4 w;
    if constexpr (k16) {
      const uint32_t x0 = St_::bits(f(8 * g)) | (St_::bits(f(8 * g + 1)) << 16);
      const uint32_t x1 = St_::bits(f(8 * g + 2)) | (St_::bits(f(8 * g + 3)) << 16);
      const uint32_t y0 = St_::bits(f(8 * g + 4)) | (St_::bits(f(8 * g + 5)) << 16);
      const uint32_t y1 = St_::bits(f(8 * g + 6)) | (St_::bits(f(8 * g + 7)) << 16);
      const auto s0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
      w = make_uint4(s0[0], s1[0], s0[1], s1[1]);
    } else {
      w = make_uint4(__float_as_uint(f(4 * g)), __float_as_uint(f(4 * g + 1)), __float_as_uint(f(4 * g + 2)),
                     __float_as_uint(f(4 * g + 3)));
    }
    return w;
  };
  auto col = [&](int g) { return k16 ? 8 * (2 * g + lh) : 8 * g + 4 * lh; };
  switch (out.a.kind) {
    case GemmEpi::Geglu:  // 16 bit only (gemm_tiles)
      if constexpr (NJ % 2 == 0 && k16) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int p = 0; p < NJ / 2; ++p)
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const uint4 w = pack(g, [&](int r) {
                return gelu16<T>(St_::rnd(acc[i][2 * p][r])) * St_::rnd(acc[i][2 * p + 1][r]);
              });
              const int m = m0 + 32 * i;
              if (m < M) *reinterpret_cast<uint4*>(C + (size_t)m * (N / 2) + nb / 2 + 32 * p + col(g)) = w;
            }
      }
      break;
    case GemmEpi::GegluSplit:  // fp32 only
      if constexpr (NJ % 2 == 0 && !k16) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int p = 0; p < NJ / 2; ++p)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              float v[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) v[r] = gelu_t<float>(acc[i][2 * p][4 * g + r]) * acc[i][2 * p + 1][4 * g + r];
              const int m = m0 + 32 * i;
              if (m < M)
                store_split4(static_cast<bf16*>(out.a.C), split_index(m, nb / 2 + 32 * p + col(g), N / 2), v);
            }
      }
      break;
    case GemmEpi::Resid: {
      uint4 old[MI][NJ][G];  // rows past M load row M - 1 (unconditional loads, issued together)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int g = 0; g < G; ++g)
            old[i][j][g] =
                *reinterpret_cast<const uint4*>(C + (size_t)min(m0 + 32 * i, M - 1) * N + nb + 32 * j + col(g));
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const uint4 w = pack(g, [&](int r) { return acc[i][j][r]; });
            const T* pw = reinterpret_cast<const T*>(&w);
            const T* po = reinterpret_cast<const T*>(&old[i][j][g]);
            uint4 res;
            T* pr = reinterpret_cast<T*>(&res);
#pragma unroll
            for (int e = 0; e < V; ++e) pr[e] = St_::st(St_::ld(po[e]) + St_::ld(pw[e]));
            const int m = m0 + 32 * i;
            if (m < M) *reinterpret_cast<uint4*>(C + (size_t)m * N + nb + 32 * j + col(g)) = res;
          }
      break;
    }
    case GemmEpi::Store:
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const uint4 w = pack(g, [&](int r) { return acc[i][j][r]; });
            const int m = m0 + 32 * i;
            if (m < M) *reinterpret_cast<uint4*>(C + (size_t)m * N + nb + 32 * j + col(g)) = w;
          }
      break;
    case GemmEpi::StoreF32:  // a caller's buffer: aligned to its element only
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int m = m0 + 32 * i;
            if (m < M)
              static_cast<float*>(out.a.C)[(size_t)m * N + nb + 32 * j + 8 * (r >> 2) + 4 * lh + (r & 3)] =
                  St_::rnd(acc[i][j][r]);
          }
      break;
    default: {  // CrossKV: column n = (layer*2 + kv)*HD + h*64 + d, row m = b*S + s
      size_t ro[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int m = m0 + 32 * i, b = m / out.a.S;
        ro[i] = (size_t)b * out.a.H * out.a.S * 64 + (size_t)(m - b * out.a.S) * 64;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {  // the 32 columns of a tile lie in one head
        const int n = nb + 32 * j, lk = n / out.a.HD, nn = n - lk * out.a.HD;
        T* base = C + ((size_t)lk * out.a.nb * out.a.H + (nn >> 6)) * out.a.S * 64 + (nn & 63);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const uint4 w = pack(g, [&](int r) { return acc[i][j][r]; });
            if (m0 + 32 * i < M) *reinterpret_cast<uint4*>(base + ro[i] + col(g)) = w;
          }
      }
    }
  }
}

// C = A B^T with the GemmOut epilogue (A (M, K), B (N, K): 16-bit rows, or split rows
// of an fp32 matrix; fp32 accumulation).  One persistent block per CU: block L
// takes tiles L, L + gridDim, .. (gridDim % 8 == 0) of the grouped_tile order.
// The k-tiles of all its tiles are one stream through the ring: while a tile's
// results are converted and stored, the next tile's first k-tiles land, and its
// multiplies start while the stores drain (vmcnt counts in order: the first wait
// of a tile leaves the previous tile's stores outstanding).  With one tile per block
// the epilogue and the refill cost 7 of 33 us at 256 x 256 x 1,024: 731 us against
// 666 us at 64,384 x 5,632 x 1,024 (1,115 TFLOP/s; operands in cache).  Rows past M read row M - 1 (not
// stored); N % BN == 0.
template <class Core, typename T, int BM, int BN, int WM, int WN, int S>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_ring(const void* __restrict__ A, const void* __restrict__ B,
                                                            int M, int N, int K, int GM, GemmOut<T> out) {
  using Tile = RingTile<Core, BM, BN, WM, WN, S>;
  extern __shared__ __align__(16) unsigned char lds[];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tm = (M + BM - 1) / BM, tn = N / BN, tiles = tm * tn, nk = K / Core::kDepth;
  const int x = blockIdx.x & 7, cnt = (tiles >> 3) + (x < (tiles & 7)), step = gridDim.x >> 3;
  const size_t ld = (size_t)nk * Tile::kRow;  // bytes of an operand row
  auto origin = [&](int i, int& m0, int& n0) {
    int mt, nt;
    grouped_tile(x + 8 * i, tm, tn, GM, mt, nt);
    m0 = mt * BM;
    n0 = nt * BN;
  };
  int t = blockIdx.x >> 3;
  if (t >= cnt) return;

  // the next k-tile to request: tile lt, depth lk; byte offsets of this thread's
  // chunks from the tile's first rows
  int lt = t, lk = 0;
  const char *ab, *bb;
  unsigned ao[Tile::LA], bo[Tile::LB];
#pragma unroll
  for (int q = 0; q < Tile::LB; ++q) {
    int row, chunk;
    Tile::load_pos(q, row, chunk);
    bo[q] = row * (unsigned)ld + chunk * 16;
  }
  auto point = [&]() {
    int m0, n0;
    origin(lt, m0, n0);
    ab = static_cast<const char*>(A) + m0 * ld;
    bb = static_cast<const char*>(B) + n0 * ld;
#pragma unroll
    for (int q = 0; q < Tile::LA; ++q) {
      int row, chunk;
      Tile::load_pos(q, row, chunk);
      ao[q] = min(row, M - 1 - m0) * (unsigned)ld + chunk * 16;
    }
  };
  point();
  auto issue = [&](unsigned char* stage) {
    const char *a = ab + (size_t)lk * Tile::kRow, *b = bb + (size_t)lk * Tile::kRow;
#pragma unroll
    for (int q = 0; q < Tile::LA; ++q) Tile::load_a(stage, q, a + ao[q]);
#pragma unroll
    for (int q = 0; q < Tile::LB; ++q) Tile::load_b(stage, q, b + bo[q]);
    if (++lk == nk) {
      if (lt + step < cnt) {
        lt += step;
        lk = 0;
        point();
      } else {
        lk = nk - 1;  // past the end: the last k-tile again, into a free stage
      }
    }
  };

  typename Tile::State s;
  Tile::start(lds, s, issue);
  // store instructions of a whole tile's epilogue: 16 bytes each, half as many for
  // the 16-bit gated-GELU pairs; three times 8 bytes for 16 of the fp32 pairs' (split)
  constexpr int kStores = Tile::MI * Tile::NJ * (sizeof(T) == 2 ? 2 : 4);
  constexpr int kGegluStores = sizeof(T) == 2 ? kStores / 2 : kStores / 2 * 3;
  const bool pairs = out.a.kind == (sizeof(T) == 2 ? GemmEpi::Geglu : GemmEpi::GegluSplit);
  const bool plain = out.a.kind == GemmEpi::Store || out.a.kind == GemmEpi::CrossKV;
  bool stored = false;  // the previous tile's epilogue issued exactly those stores after the ring's loads
  for (; t < cnt; t += step) {
    int m0, n0;
    origin(t, m0, n0);
    s.clear();
    Tile::reread(lds, s);  // the first fragments need no registers across the epilogue
    for (int kt = 0; kt < nk; ++kt) {
      const bool after = stored && kt == 0;
      Tile::ktile(lds, s, issue, [&] {
        if (after && plain)
          Tile::template wait_loads<kStores>();
        else if (after && pairs)
          Tile::template wait_loads<kGegluStores>();
        else
          Tile::template wait_loads<>();
      });
    }
    s.settle();
    if constexpr (sizeof(T) == 4)
      resum_not_finite<Tile>(s, [&](int row, int col) {
        return split_dot(reinterpret_cast<const bf16*>(static_cast<const char*>(A) + min(m0 + row, M - 1) * ld),
                         reinterpret_cast<const bf16*>(static_cast<const char*>(B) + (n0 + col) * ld), nk, 0.f);
      });
    mfma_epilogue<T, Tile::MI, Tile::NJ>(out, s.acc, M, m0 + (wid / WN) * (BM / WM), n0 + (wid % WN) * (BN / WN));
    asm volatile("" ::: "memory");  // the stores stay ahead of the next tile's waits
    stored = m0 + BM <= M;
  }
  __builtin_amdgcn_s_waitcnt(vm_wait_imm(0));  // no copy into LDS outlives the block
}

template <class Core, typename T, int BM, int BN, int WM, int WN, int S>
void launch_gemm_ring(const void* A, const void* B, int M, int N, int K, const GemmOut<T>& out, hipStream_t s) {
  using Tile = RingTile<Core, BM, BN, WM, WN, S>;
  const auto kernel = &k_gemm_ring<Core, T, BM, BN, WM, WN, S>;
  allow_dynamic_lds(reinterpret_cast<const void*>(kernel), Tile::kLds);
  const long tiles = (long)((M + BM - 1) / BM) * (N / BN);
  MRT_REQUIRE(N % BN == 0 && K % Core::kDepth == 0 && tiles <= 0x7fffffffL, "gemm: tile does not fit the shape");
  MRT_REQUIRE((long)K / Core::kDepth * Tile::kRow * (BM > BN ? BM : BN) <= 0xffffffffL, "gemm: rows too long");
  const long grid = std::min((long)std::max(8, device_cus() & ~7), (tiles + 7) / 8 * 8);
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(Tile::kThreads), Tile::kLds, s, A, B, M, N, K, 4, out);
}

// ---- encoder self-attention (bidirectional, no mask, no bias, scale 1.0) -------------
// One lane per query row, 64 rows per block; K/V tiles of 64 keys staged in
// LDS; online softmax per 64-key tile.
template <typename T>
__global__ __launch_bounds__(64) void k_enc_attn(const T* __restrict__ qkv, int S, int H,
                                                 T* __restrict__ out) {
  using St_ = St<T>;
  const int bh = blockIdx.y, b = bh / H, h = bh - b * H, lane = threadIdx.x;
  const int HD = H * 64, ld = 3 * HD;
  const int qi = blockIdx.x * 64 + lane;
  __shared__ float Ks[64][64 + 1];
  __shared__ float Vs[64][64];
  float q[64], o[64];
  const T* qrow = qkv + ((size_t)b * S + (qi < S ? qi : 0)) * ld + h * 64;
#pragma unroll
  for (int d = 0; d < 64; ++d) {
    q[d] = St_::ld(qrow[d]);
    o[d] = 0.f;
  }
  float m = -INFINITY, l = 0.f;
  for (int j0 = 0; j0 < S; j0 += 64) {
    const int nk = min(64, S - j0);
    for (int r = 0; r < nk; ++r) {
      const T* row = qkv + ((size_t)b * S + j0 + r) * ld + h * 64;
      Ks[r][lane] = St_::ld(row[HD + lane]);
      Vs[r][lane] = St_::ld(row[2 * HD + lane]);
    }
    for (int r = nk; r < 64; ++r) Vs[r][lane] = 0.f;  // met by zero weights: LDS may hold NaN
    __syncthreads();
    float sc[64];
    float mt = -INFINITY;
#pragma unroll
    for (int r = 0; r < 64; ++r) {
      float acc = 0.f;
#pragma unroll
      for (int d = 0; d < 64; ++d) acc = fmaf(q[d], Ks[r][d], acc);
      sc[r] = r < nk ? acc : -INFINITY;
      mt = fmaxf(mt, sc[r]);
    }
    const float mn = fmaxf(m, mt);
    const float corr = expf(m - mn);
    l *= corr;
#pragma unroll
    for (int d = 0; d < 64; ++d) o[d] *= corr;
#pragma unroll
    for (int r = 0; r < 64; ++r) {
      const float p = r < nk ? expf(sc[r] - mn) : 0.f;
      l += p;
#pragma unroll
      for (int d = 0; d < 64; ++d) o[d] = fmaf(p, Vs[r][d], o[d]);
    }
    m = mn;
    __syncthreads();
  }
  if (qi < S) {
    T* orow = out + ((size_t)b * S + qi) * HD + h * 64;
    const float inv = 1.0f / l;
#pragma unroll
    for (int d = 0; d < 64; ++d) orow[d] = St_::st(o[d] * inv);
  }
}

// ---- 16-bit encoder self-attention on MFMA ------------------------------------------
// Flash attention for one (row, head) and 128 queries per workgroup (32 per
// wave), keys in tiles of 64 staged in LDS.  Scores are computed transposed,
// S^T = K Q^T (v_mfma_f32_32x32x16_{bf16,f16}), so lane l owns query l % 32 and
// the online-softmax rescale is per lane.  The output is also accumulated
// transposed, O^T += V^T P^T, with P^T taken straight from the score
// accumulators: lane l's accumulators of a 16-key step hold keys
// {4h..4h+3, 8+4h..8+4h+3} (h = l / 32), so V^T is staged with the key order
// inside every 16-key block permuted the same way (swap of key bits 2 and 3).
// Scores and the softmax are fp32, the exponentials taken as
// 2^(s log2 e - m log2 e) with one fma and v_exp_f32 (as fused attention
// kernels do), keys past S masked only in the last tile; P enters the second
// product as the sum of two parts in the storage type (hi + lo: ~16
// significant bits for bf16, ~22 for fp16), as close to the fp32
// probabilities of the reference's fused attention as 16-bit MFMA allows (P
// rounded once to bf16 measured 2.02e-2 on a level slice of the bf16
// two-frame decode against the oracle's 2e-2 bound).
constexpr int kAQ = 128, kAK = 64, kALD = 64 + 8;  // queries, keys per tile, padded LDS row
constexpr float kLog2e = 1.4426950408889634f;

// Element offset of 8-key chunk `ch` in row `dim` of the staged V^T: chunks are
// XOR-swizzled by dim / 8, so the transposed 2-byte stores of 8 dims 8 apart
// fall in different banks (2-way instead of 8-way), while the padded rows keep
// the 16-byte fragment reads of 8 consecutive dims conflict-free.
__device__ __forceinline__ int vt_chunk(int ch, int dim) { return (ch ^ ((dim >> 3) & 7)) << 3; }

// Scores of one 64-key tile from the staged K rows: sc[t] holds S^T for keys
// 32 t + 8 (r / 4) + 4 hf + r % 4 of the tile, query lq.
template <typename T>
__device__ __forceinline__ void attn_scores(const T* Ks, const typename Mfma<T>::v8 (&qf)[4], int lq, int hf,
                                            f32x16_t (&sc)[2]) {
  typedef typename Mfma<T>::v8 v8;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[t][r] = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const v8 a = *reinterpret_cast<const v8*>(&Ks[(32 * t + lq) * kALD + 16 * s + 8 * hf]);
      sc[t] = Mfma<T>::mma(a, qf[s], sc[t]);
    }
  }
}

// Online-softmax step of one tile (keys kb ..): running max m, sum lsum and
// output accumulators acc, with the tile's V^T staged in Vt.
template <typename T>
__device__ __forceinline__ void attn_update(f32x16_t (&sc)[2], int kb, int S, int lq, int hf, const T* Vt, float& m,
                                            float& lsum, f32x16_t (&acc)[2]) {
  typedef typename Mfma<T>::v8 v8;
  float mt = -INFINITY;
  if (kb + kAK <= S) {  // a full tile (wave-uniform): no key to mask
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sc[t][r]);
  } else {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kb + 32 * t + 8 * (r >> 2) + 4 * hf + (r & 3);
        sc[t][r] = key < S ? sc[t][r] : -INFINITY;
        mt = fmaxf(mt, sc[t][r]);
      }
  }
  mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
  const float mn = fmaxf(m, mt);  // raw-score running max (key 0 is never masked)
  const float mns = mn * kLog2e;
  const float corr = __builtin_amdgcn_exp2f(fmaf(m, kLog2e, -mns));
  float ps = 0.f;
  v8 pb[4], pl[4];  // P^T = hi + lo (storage type each) for the four 16-key steps
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    f32x8_t pv;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pv[i] = __builtin_amdgcn_exp2f(fmaf(sc[g >> 1][8 * (g & 1) + i], kLog2e, -mns));
      ps += pv[i];
    }
    pb[g] = __builtin_convertvector(pv, v8);  // round-to-nearest-even conversions
    pl[g] = __builtin_convertvector(pv - __builtin_convertvector(pb[g], f32x8_t), v8);
  }
  ps += __shfl_xor(ps, 32, 64);
  lsum = lsum * corr + ps;
  m = mn;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] *= corr;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const v8 a = *reinterpret_cast<const v8*>(&Vt[(32 * t + lq) * kALD + vt_chunk(2 * s + hf, 32 * t + lq)]);
      acc[t] = Mfma<T>::mma(a, pb[s], acc[t]);
      acc[t] = Mfma<T>::mma(a, pl[s], acc[t]);
    }
}

// Tile j + 1's K and V are loaded (K rows first, then V rows) while tile j is
// processed.  Sized for three blocks per CU (3 waves per SIMD: the register
// budget is 170), which measured faster than the compiler's 196 registers at
// two.  Every query runs attn_scores / attn_update over the tiles in order,
// the same arithmetic whatever the grid, so a stream's rows do not depend on
// the batch it is encoded in.
template <typename T>
__global__ __launch_bounds__(256, 3) void k_enc_attn_mfma(const T* __restrict__ qkv, int S, int H,
                                                       T* __restrict__ out) {
  typedef typename Mfma<T>::v8 v8;
  __shared__ __attribute__((aligned(16))) T Ks[2][kAK * kALD];
  __shared__ __attribute__((aligned(16))) T Vt[2][64 * kALD];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int bh = blockIdx.y, b = bh / H, h = bh - b * H;
  const int HD = H * 64, ld = 3 * HD;
  const T* base = qkv + (size_t)b * S * ld + h * 64;
  const int lq = lane & 31, hf = lane >> 5;
  const int q = blockIdx.x * kAQ + wid * 32 + lq;

  // Q^T fragments (B operand): lane l holds Q[q][16 s + 8 hf .. +7].
  v8 qf[4];
  {
    const T* qr = base + (size_t)min(q, S - 1) * ld;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = *reinterpret_cast<const v8*>(qr + 16 * s + 8 * hf);
  }
  // Tile staging: thread t moves 16 bytes of K (part 1 of the q/k/v row) or V
  // (part 2) for keys t/8 and 32 + t/8, dims 8 (t % 8) .. +7; keys past S are
  // zero.  (Clamping those keys to S - 1 instead, with no conditional load,
  // made the compiler keep the Q fragments in scratch memory.)
  uint4 rk[2], rv[2];
  auto gload = [&](uint4 (&r)[2], int kb, int part) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = kb + (tid >> 3) + 32 * i, c = (tid & 7) * 8;
      r[i] = key < S ? *reinterpret_cast<const uint4*>(base + (size_t)key * ld + part * HD + c)
                     : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  auto kstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = (tid >> 3) + 32 * i, c = (tid & 7) * 8;
      *reinterpret_cast<uint4*>(&Ks[buf][key * kALD + c]) = rk[i];
    }
  };
  auto vstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = (tid >> 3) + 32 * i, c = (tid & 7) * 8;
      const int slot = (key & ~12) | ((key & 4) << 1) | ((key & 8) >> 1);
      const T* v = reinterpret_cast<const T*>(&rv[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) Vt[buf][(c + e) * kALD + vt_chunk(slot >> 3, c + e) + (slot & 7)] = v[e];
    }
  };

  f32x16_t acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  float m = -INFINITY, lsum = 0.f;
  const int ntiles = (S + kAK - 1) / kAK;

  gload(rk, 0, 1);
  gload(rv, 0, 2);
  kstore(0);
  vstore(0);
  __syncthreads();
  for (int j = 0; j < ntiles; ++j) {
    const int cur = j & 1, kb = j * kAK;
    if (j + 1 < ntiles) {
      gload(rk, kb + kAK, 1);
      gload(rv, kb + kAK, 2);
    }
    f32x16_t sc[2];
    attn_scores<T>(Ks[cur], qf, lq, hf, sc);
    attn_update<T>(sc, kb, S, lq, hf, Vt[cur], m, lsum, acc);
    if (j + 1 < ntiles) {
      kstore(cur ^ 1);
      vstore(cur ^ 1);
    }
    __syncthreads();
  }
  if (q < S) {
    T* orow = out + ((size_t)b * S + q) * HD + h * 64;
    const float inv = 1.0f / lsum;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * t + 8 * g + 4 * hf;
        uint2 w;
        w.x = St<T>::bits(acc[t][4 * g] * inv) | (St<T>::bits(acc[t][4 * g + 1] * inv) << 16);
        w.y = St<T>::bits(acc[t][4 * g + 2] * inv) | (St<T>::bits(acc[t][4 * g + 3] * inv) << 16);
        *reinterpret_cast<uint2*>(orow + d) = w;
      }
  }
}

}  // namespace

void encoder_embed(DType dt, const void* emb, const void* pe, const int* tok, int M, int S, int D,
                   void* x, hipStream_t s) {
  MRT_DTYPE_DISPATCH(dt, hipLaunchKernelGGL(k_encoder_embed<T>, dim3(M), dim3(256), 0, s, (const T*)emb,
                                            (const T*)pe, tok, S, D, (T*)x));
  MRT_HIP_CHECK(hipGetLastError());
}

namespace {

// The wave-per-row norm for rows of 64 V NV elements (NV <= 4) on 16-byte
// aligned pointers; false when the shape or alignment does not fit.
template <typename T, bool FRAG>
bool rmsnorm_rows_wave(const T* x, const T* g, float eps, int M, int D, T* y, hipStream_t s) {
  constexpr int W = 64 * St<T>::kVec;
  const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(g) |
                         reinterpret_cast<uintptr_t>(y)) & 15) == 0;
  if (!aligned || D % W != 0 || D / W < 1 || D / W > 4) return false;
  const dim3 grid((M + 3) / 4), block(256);
  switch (D / W) {
    case 1: hipLaunchKernelGGL((k_rmsnorm_rows_wave<T, 1, FRAG>), grid, block, 0, s, x, g, eps, M, D, y); break;
    case 2: hipLaunchKernelGGL((k_rmsnorm_rows_wave<T, 2, FRAG>), grid, block, 0, s, x, g, eps, M, D, y); break;
    case 3: hipLaunchKernelGGL((k_rmsnorm_rows_wave<T, 3, FRAG>), grid, block, 0, s, x, g, eps, M, D, y); break;
    default: hipLaunchKernelGGL((k_rmsnorm_rows_wave<T, 4, FRAG>), grid, block, 0, s, x, g, eps, M, D, y); break;
  }
  return true;
}

template <typename T, bool FRAG>
void rmsnorm_rows_t(const void* xv, const void* gv, float eps, int M, int D, void* yv, hipStream_t s) {
  const T *x = static_cast<const T*>(xv), *g = static_cast<const T*>(gv);
  T* y = static_cast<T*>(yv);
  if (rmsnorm_rows_wave<T, FRAG>(x, g, eps, M, D, y, s)) return;
  hipLaunchKernelGGL((D <= 256 * kNormPer ? k_rmsnorm_rows_reg<T, FRAG> : k_rmsnorm_rows<T, FRAG>), dim3(M), dim3(256),
                     0, s, x, g, eps, D, y);
}

}  // namespace

void rmsnorm_rows(DType dt, const void* x, const void* g, float eps, int M, int D, void* y, hipStream_t s,
                  bool frag_out) {
  if (frag_out) {
    MRT_REQUIRE(dt != DType::F32 && D % 32 == 0, "norm: fragments hold 16-bit rows of whole 32 columns");
    if (dt == DType::BF16)
      rmsnorm_rows_t<bf16, true>(x, g, eps, M, D, y, s);
    else
      rmsnorm_rows_t<f16, true>(x, g, eps, M, D, y, s);
  } else {
    MRT_DTYPE_DISPATCH(dt, (rmsnorm_rows_t<T, false>(x, g, eps, M, D, y, s)));
  }
  MRT_HIP_CHECK(hipGetLastError());
}

namespace {

// The tiles, in the order in which they are preferred, with their time per area
// relative to the first.
struct GemmTile {
  int bm, bn;
  double f;
};
constexpr GemmTile kTiles16[] = {{256, 256, 1.0}, {192, 256, 1.03}, {128, 256, 1.14}, {128, 192, 1.24}, {64, 128, 2.0}};
constexpr GemmTile kTiles32[] = {{128, 192, 1.0}, {128, 128, 1.06}, {64, 128, 1.22}};

bool gemm_pairs(GemmEpi kind) { return kind == GemmEpi::Geglu || kind == GemmEpi::GegluSplit; }

// Gated-GELU pairs need wave tiles of whole 64-column groups (not 192 columns).
bool tile_takes(const GemmTile& t, int N, GemmEpi kind) { return N % t.bn == 0 && !(gemm_pairs(kind) && t.bn == 192); }

// The tile whose rounds over the CUs (one block each) take the least time: rounds x
// area x the tile's time per area.  The factors are measured: three rounds on 256
// CUs, operands from memory, us, 16 bit at K = 1,024 and 2,816: 256 x 256 106 and 248;
// 192 x 256 84.3 and 193; 128 x 256 61.9 and 142; 128 x 192 49.4 and 115; 64 x 128
// 27.2 and 60.8 (its fragment reads and its epilogue weigh more); fp32: 128 x 192 190
// and 507; 128 x 128 137 and 353; 64 x 128 80.7 and 196.  The residual and gated
// epilogues leave the ratios as they are within 6 %.
template <int n>
int best_tile(const GemmTile (&tiles)[n], int M, int N, GemmEpi kind) {
  const long cus = std::max(8, device_cus() & ~7);
  int best = -1;
  double least = 0.;
  for (int i = 0; i < n; ++i) {
    const GemmTile& t = tiles[i];
    if (!tile_takes(t, N, kind)) continue;
    const long count = (long)((M + t.bm - 1) / t.bm) * (N / t.bn);
    const double cost = (double)((count + cus - 1) / cus) * t.bm * t.bn * t.f;
    if (best < 0 || cost < least) best = i, least = cost;
  }
  return best;
}

}  // namespace

int gemm_tile(DType dt, int M, int N, GemmEpi kind) {
  return dt == DType::F32 ? best_tile(kTiles32, M, N, kind) : best_tile(kTiles16, M, N, kind);
}

namespace {

template <class Core, typename T>
void gemm_tiles(const void* A, const void* B, int M, int N, int K, const GemmEpiArgs& e, hipStream_t s) {
  const GemmOut<T> out{e, N};
  const int tile = e.tile >= 0 ? e.tile : gemm_tile(sizeof(T) == 2 ? DType::BF16 : DType::F32, M, N, e.kind);
  if constexpr (sizeof(T) == 2) {
    MRT_REQUIRE(tile >= 0 && tile < 5 && tile_takes(kTiles16[tile], N, e.kind), "gemm: tile does not fit the shape");
    switch (tile) {
      case 0: launch_gemm_ring<Core, T, 256, 256, 4, 2, 2>(A, B, M, N, K, out, s); break;
      case 1: launch_gemm_ring<Core, T, 192, 256, 2, 4, 2>(A, B, M, N, K, out, s); break;
      case 2: launch_gemm_ring<Core, T, 128, 256, 2, 4, 3>(A, B, M, N, K, out, s); break;
      case 3: launch_gemm_ring<Core, T, 128, 192, 4, 2, 3>(A, B, M, N, K, out, s); break;
      default: launch_gemm_ring<Core, T, 64, 128, 2, 2, 4>(A, B, M, N, K, out, s); break;
    }
  } else {
    MRT_REQUIRE(e.kind != GemmEpi::Geglu, "gemm: fp32 pairs are written split");
    MRT_REQUIRE(tile >= 0 && tile < 3 && tile_takes(kTiles32[tile], N, e.kind), "gemm: tile does not fit the shape");
    switch (tile) {
      case 0: launch_gemm_ring<Core, T, 128, 192, 2, 2, 2>(A, B, M, N, K, out, s); break;
      case 1: launch_gemm_ring<Core, T, 128, 128, 2, 2, 3>(A, B, M, N, K, out, s); break;
      default: launch_gemm_ring<Core, T, 64, 128, 2, 2, 4>(A, B, M, N, K, out, s); break;
    }
  }
}

template <typename T>
void gemm_t(const T* A, const T* B, int M, int N, int K, const GemmEpiArgs& e, hipStream_t s, bool allow_mfma) {
  GemmOut<T> out{e, N};
  if constexpr (sizeof(T) == 2) {
    if (allow_mfma && N % 128 == 0 && K % 64 == 0) {
      gemm_tiles<Core16<T>, T>(A, B, M, N, K, e, s);
      return;
    }
  }
  hipLaunchKernelGGL(k_gemm_valu<T>, dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, s, A, B, M, N, K, out);
}

}  // namespace

void gemm(DType dt, const void* A, const void* B, int M, int N, int K, const GemmEpiArgs& e,
          hipStream_t s, bool allow_mfma) {
  MRT_REQUIRE(M >= 1 && N >= 1 && K >= 1, "gemm: empty problem");
  MRT_REQUIRE(e.kind != GemmEpi::GegluSplit, "gemm: split pairs come from split operands");
  if (e.kind == GemmEpi::Geglu) MRT_REQUIRE(N % 64 == 0, "gemm: gated-GELU needs N % 64 == 0");
  if (e.kind == GemmEpi::CrossKV)
    MRT_REQUIRE(e.HD == e.H * 64 && N % e.HD == 0 && M == e.nb * e.S, "gemm: bad cross-KV shape");
  MRT_DTYPE_DISPATCH(dt, gemm_t<T>(static_cast<const T*>(A), static_cast<const T*>(B), M, N, K, e, s, allow_mfma));
  MRT_HIP_CHECK(hipGetLastError());
}

bool gemm_split_fits(int N, int K) { return N % 128 == 0 && K % 32 == 0 && K >= 32; }

void gemm_split(const bf16* A, const bf16* B, int M, int N, int K, const GemmEpiArgs& e, hipStream_t s) {
  MRT_REQUIRE(M >= 1 && gemm_split_fits(N, K), "split gemm: N must be a multiple of 128, K of 32");
  if (e.kind == GemmEpi::CrossKV)
    MRT_REQUIRE(e.HD == e.H * 64 && N % e.HD == 0 && M == e.nb * e.S, "gemm: bad cross-KV shape");
  gemm_tiles<CoreSplitFine, float>(A, B, M, N, K, e, s);
  MRT_HIP_CHECK(hipGetLastError());
}

namespace {

template <typename T>
void encoder_attn_t(const T* qkv, int nb, int S, int H, T* out, hipStream_t s, bool allow_mfma) {
  if constexpr (sizeof(T) == 2) {
    if (allow_mfma) {
      hipLaunchKernelGGL(k_enc_attn_mfma<T>, dim3((S + kAQ - 1) / kAQ, nb * H), dim3(256), 0, s, qkv, S, H, out);
      return;
    }
  }
  hipLaunchKernelGGL(k_enc_attn<T>, dim3((S + 63) / 64, nb * H), dim3(64), 0, s, qkv, S, H, out);
}

}  // namespace

void encoder_attn(DType dt, const void* qkv, int nb, int S, int H, void* out, hipStream_t s, bool allow_mfma) {
  MRT_DTYPE_DISPATCH(dt, encoder_attn_t<T>(static_cast<const T*>(qkv), nb, S, H, static_cast<T*>(out), s, allow_mfma));
  MRT_HIP_CHECK(hipGetLastError());
}

}  // namespace mrt
