// Kernels around the split fp32 GEMM (split_gemm.hpp) of the fp32 encoder: the
// split of row-major matrices, the RMSNorm that writes split rows, and the
// encoder's self-attention on the fp32 matrix instruction.
#include "kernels.hpp"
#include "split_gemm.hpp"

namespace mrt {
namespace {

// W may be a caller's tensor, aligned to its element only (global loads of 16 bytes
// need no more).
__global__ __launch_bounds__(256) void k_split_rows(const float* __restrict__ W, size_t n4, bf16* __restrict__ out) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
    const f4 v = reinterpret_cast<const f4*>(W)[i];
    const size_t e = 4 * i;  // rows are whole groups, so groups run through the matrix
    store_split4(out, (e >> 5) * kSplitGroup + (e & 31), {v.x, v.y, v.z, v.w});
  }
}

// One wave per row of D = 256 NV floats or fewer (D % 32 == 0), as the 16-bit
// row norm: a lane keeps its chunks of 4 between the sum of squares and the
// scaling.
template <int NV>
__global__ __launch_bounds__(256) void k_rmsnorm_split(const float* __restrict__ x, const float* __restrict__ g,
                                                       float eps, int M, int D, bf16* __restrict__ y) {
  const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);  // wave-uniform
  if (r >= M) return;
  const int nch = D / 4;
  const float4* xr = reinterpret_cast<const float4*>(x + (size_t)r * D);
  const float4* gr = reinterpret_cast<const float4*>(g);
  float4 v[NV], gv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = min(lane + 64 * i, nch - 1);
    v[i] = xr[c];
    gv[i] = gr[c];
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if (lane + 64 * i < nch) ss += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if (lane + 64 * i < nch)
      store_split4(y, split_index(r, 4 * (lane + 64 * i), D),
                   {v[i].x * inv * gv[i].x, v[i].y * inv * gv[i].y, v[i].z * inv * gv[i].z, v[i].w * inv * gv[i].w});
}

// fp32 flash attention on v_mfma_f32_32x32x2_f32: one (row, head) and 128
// queries per workgroup of 8 waves.  Wave w takes queries 32 (w % 4) .. + 31 over
// the even (w < 4) or odd 64-key tiles, and the two halves' softmax states meet
// in LDS at the end: 256 workgroups of one stream then give every SIMD two
// waves, one of which multiplies while the other exponentiates.  K and V of a
// tile pair are staged in double-buffered LDS.
//
// Scores are computed transposed, S^T = K Q^T, so a lane owns query lane % 32
// and the online softmax is per lane; the output accumulates O^T += V^T P^T.
// The instruction multiplies two k a step, one per lane half: the score steps
// take dims 8 u + e and 8 u + 4 + e (one 16-byte read of a K row feeds four
// steps), the output steps keys k and k + 4 of a group of 8, which is where the
// score accumulators hold P, so P never leaves its registers and V is read as
// it is stored.  Softmax in fp32 with expf, P unrounded.  128 instructions of
// 64 cycles a tile and wave bound it: 56 us a layer of 2 x 16 heads x 1006
// queries at the instruction's rate.  Measured: one lane per query on the vector
// ALUs 1,472 us, one wave per SIMD over all tiles 138 us, this 97 us.
constexpr int kFaQ = 128, kFaK = 64, kFaKLd = 64 + 4;  // queries, keys per tile, padded K row
constexpr int kFaPair = 2 * kFaK;                      // keys staged at a time
constexpr size_t kFaLds = 2 * sizeof(float) * kFaPair * (kFaKLd + 64);
constexpr int kFaMerge = 34;                           // floats a lane hands over: 32 outputs, maximum, sum

__global__ __launch_bounds__(512) void k_enc_attn_f32(const float* __restrict__ qkv, int S, int H,
                                                      bf16* __restrict__ out) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  extern __shared__ __align__(16) float fa_lds[];
  constexpr int kBuf = kFaPair * (kFaKLd + 64), kV = kFaPair * kFaKLd;  // a buffer: K rows, then V rows
  // scalar wave index: matrix instructions ignore the lane mask
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wid >> 2;
  const int bh = blockIdx.y, b = bh / H, h = bh - b * H;
  const int HD = H * 64, ld = 3 * HD;
  const float* base = qkv + (size_t)b * S * ld + h * 64;
  const int lq = lane & 31, hf = lane >> 5;
  const int q = blockIdx.x * kFaQ + (wid & 3) * 32 + lq;

  float qf[32];  // Q[q][8 u + 4 hf + e] at 4 u + e
  {
    const float* qr = base + (size_t)min(q, S - 1) * ld;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float4 v = *reinterpret_cast<const float4*>(qr + 8 * u + 4 * hf);
      qf[4 * u] = v.x;
      qf[4 * u + 1] = v.y;
      qf[4 * u + 2] = v.z;
      qf[4 * u + 3] = v.w;
    }
  }
  // thread t moves 16 bytes of K and of V of keys t / 16 + 32 i, dims 4 (t % 16);
  // keys past S repeat the last (their scores are masked)
  f4 rk[4], rv[4];
  const int c4 = (tid & 15) * 4;
  auto gload = [&](int kb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* row = base + (size_t)min(kb + (tid >> 4) + 32 * i, S - 1) * ld + c4;
      rk[i] = *reinterpret_cast<const f4*>(row + HD);
      rv[i] = *reinterpret_cast<const f4*>(row + 2 * HD);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = (tid >> 4) + 32 * i;
      *reinterpret_cast<f4*>(fa_lds + buf * kBuf + key * kFaKLd + c4) = rk[i];
      *reinterpret_cast<f4*>(fa_lds + buf * kBuf + kV + key * 64 + c4) = rv[i];
    }
  };
  f32x16_t acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  float m = -INFINITY, lsum = 0.f;
  const int npairs = (S + kFaPair - 1) / kFaPair;
  gload(0);
  store(0);
  // Q has landed here: else the loop would wait for it behind its own prefetch
#pragma unroll
  for (int i = 0; i < 32; ++i) asm volatile("" : "+v"(qf[i]));
  __syncthreads();
  for (int j = 0; j < npairs; ++j) {
    const int cur = j & 1, kb = j * kFaPair + grp * kFaK;
    if (j + 1 < npairs) gload((j + 1) * kFaPair);
    if (kb < S) {
      const float* Ks = fa_lds + cur * kBuf + grp * kFaK * kFaKLd;
      const float* Vs = fa_lds + cur * kBuf + kV + grp * kFaK * 64;
      f32x16_t sc[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[t][r] = 0.f;
      f4 kv[2][2];
      auto kread = [&](int u, f4 (&d)[2]) {
#pragma unroll
        for (int t = 0; t < 2; ++t) d[t] = *reinterpret_cast<const f4*>(Ks + (32 * t + lq) * kFaKLd + 8 * u + 4 * hf);
      };
      kread(0, kv[0]);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (u < 7) kread(u + 1, kv[(u + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            sc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[u & 1][t][e], qf[4 * u + e], sc[t], 0, 0, 0);
      }
      // accumulator r of sc[t]: key 32 t + 8 (r / 4) + 4 hf + r % 4 of the tile
      if (kb + kFaK > S) {  // the last tile: keys past S
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kb + 32 * t + 8 * (r >> 2) + 4 * hf + (r & 3) >= S) sc[t][r] = -INFINITY;
      }
      float mt = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sc[t][r]);
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
      const float mn = fmaxf(m, mt);  // a tile that is run holds at least one key
      const float corr = expf(m - mn);
      m = mn;
      float ps = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          sc[t][r] = expf(sc[t][r] - mn);
          ps += sc[t][r];
        }
      ps += __shfl_xor(ps, 32, 64);
      lsum = lsum * corr + ps;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] *= corr;
      // groups of 4 keys a lane half (accumulators 4 (g % 4) .. + 3 of sc[g / 4]),
      // a group's V read while the one before is multiplied
      float v[2][4][2];
      auto vread = [&](int g, float (&d)[4][2]) {
        const float* vr = Vs + (8 * g + 4 * hf) * 64 + lq;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          d[e][0] = vr[64 * e];
          d[e][1] = vr[64 * e + 32];
        }
      };
      vread(0, v[0]);
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        if (g < 7) vread(g + 1, v[(g + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int d = 0; d < 2; ++d)
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[g & 1][e][d], sc[g >> 2][4 * (g & 3) + e], acc[d], 0, 0, 0);
      }
    }
    if (j + 1 < npairs) store(cur ^ 1);
    __syncthreads();
  }
  // the odd tiles' state joins the even tiles' (every LDS read of the loop is past the barrier)
  float* mg = fa_lds + (size_t)((wid & 3) * 64 + lane) * kFaMerge;
  if (grp == 1) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mg[16 * t + r] = acc[t][r];
    mg[32] = m;
    mg[33] = lsum;
  }
  __syncthreads();
  if (grp == 1 || q >= S) return;
  const float m1 = mg[32], mm = fmaxf(m, m1);
  const float w0 = expf(m - mm), w1 = expf(m1 - mm);  // no odd tile: m1 = -inf, w1 = 0
  const float inv = 1.0f / (lsum * w0 + mg[33] * w1);
  // accumulator r of acc[t]: dim 32 t + 8 (r / 4) + 4 hf + r % 4
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (acc[t][4 * g + e] * w0 + mg[16 * t + 4 * g + e] * w1) * inv;
      store_split4(out, split_index((size_t)b * S + q, h * 64 + 32 * t + 8 * g + 4 * hf, HD), o);
    }
}

}  // namespace

void split_rows(const float* W, long N, int K, bf16* out, hipStream_t s) {
  MRT_REQUIRE(N >= 1 && K >= 32 && K % 32 == 0, "split rows: K must be a multiple of 32");
  const size_t n4 = static_cast<size_t>(N) * K / 4;
  const int blocks = static_cast<int>(n4 / 256 + 1 < 8192 ? n4 / 256 + 1 : 8192);
  hipLaunchKernelGGL(k_split_rows, dim3(blocks), dim3(256), 0, s, W, n4, out);
  MRT_HIP_CHECK(hipGetLastError());
}

void split_upload(const float* W, long N, int K, bf16* out, hipStream_t s) {
  void* d = nullptr;
  const size_t bytes = (size_t)N * K * 4;
  MRT_HIP_CHECK(hipMalloc(&d, bytes));
  hipError_t e = hipMemcpy(d, W, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    split_rows(static_cast<const float*>(d), N, K, out, s);
    e = hipStreamSynchronize(s);
  }
  (void)hipFree(d);
  MRT_HIP_CHECK(e);
}

void rmsnorm_rows_split(const float* x, const float* g, float eps, int M, int D, bf16* y, hipStream_t s) {
  MRT_REQUIRE(M >= 1 && D % 32 == 0 && D <= 4096, "split norm: D must be a multiple of 32, at most 4096");
  const dim3 grid((M + 3) / 4), block(256);
  if (D <= 1024)
    hipLaunchKernelGGL(k_rmsnorm_split<4>, grid, block, 0, s, x, g, eps, M, D, y);
  else
    hipLaunchKernelGGL(k_rmsnorm_split<16>, grid, block, 0, s, x, g, eps, M, D, y);
  MRT_HIP_CHECK(hipGetLastError());
}

void encoder_attn_split(const float* qkv, int nb, int S, int H, bf16* out, hipStream_t s) {
  static_assert(kFaLds <= 160 * 1024 && 4 * 64 * kFaMerge * sizeof(float) <= kFaLds, "LDS of one CU");
  allow_dynamic_lds(reinterpret_cast<const void*>(&k_enc_attn_f32), kFaLds);
  hipLaunchKernelGGL(k_enc_attn_f32, dim3((S + kFaQ - 1) / kFaQ, nb * H), dim3(512), kFaLds, s, qkv, S, H, out);
  MRT_HIP_CHECK(hipGetLastError());
}

}  // namespace mrt
