// MusicCoCa text-path kernels (fp32): embedding, LayerNorm, the attention
// core and RVQ quantisation.  The projections run on the codec's matrix-core
// GEMM (conv_split.hip; codec_kernels.hip for widths it does not take).
#include "coca.hpp"
#include "device_utils.hpp"
#include "split_gemm.hpp"

namespace mrt {
namespace {

constexpr int kT = 256;

__device__ __forceinline__ float block_sum(float v, float* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
  return s;
}

__device__ __forceinline__ float block_max(float v, float* red) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  float s = red[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) s = fmaxf(s, red[i]);
  return s;
}

// musiccoca.cpp:272-277: x = table[id] * sqrt(d_model).
__global__ void k_coca_embed(const int* __restrict__ ids, const float* __restrict__ table, int vocab, int D, float scale,
                             float* __restrict__ x) {
  int id = ids[blockIdx.x];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  for (int d = threadIdx.x; d < D; d += blockDim.x) x[(size_t)blockIdx.x * D + d] = table[(size_t)id * D + d] * scale;
}

// musiccoca.cpp:71-79: mean, centred, variance of the centred values, then
// centred * rsqrt(var + eps) * w + b.  One workgroup per row.
__global__ __launch_bounds__(kT) void k_layer_norm(const float* __restrict__ x, int D, const float* __restrict__ w,
                                                   const float* __restrict__ b, float eps, float* __restrict__ y,
                                                   bf16* __restrict__ ys) {
  __shared__ float red[kT / 64];
  const float* xr = x + (size_t)blockIdx.x * D;
  float s = 0.f;
  for (int d = threadIdx.x; d < D; d += kT) s += xr[d];
  const float mean = block_sum(s, red) / (float)D;
  float v = 0.f;
  for (int d = threadIdx.x; d < D; d += kT) {
    const float c = xr[d] - mean;
    v += c * c;
  }
  const float var = block_sum(v, red) / (float)D;
  const float inv = rsqrtf(var + eps);
  for (int d = threadIdx.x; d < D; d += kT) {
    const float o = (xr[d] - mean) * inv * w[d] + b[d];
    if (ys)
      store_split(ys, split_index(blockIdx.x, d, D), o);
    else
      y[(size_t)blockIdx.x * D + d] = o;
  }
}

// One workgroup per (query, head): thread j < Sk scores key j, the softmax
// runs over the workgroup, then threads split the head's D outputs.
__global__ __launch_bounds__(kT) void k_coca_attention(const float* __restrict__ q, int ldq,
                                                       const float* __restrict__ k, int ldk,
                                                       const float* __restrict__ v, int ldv, int Sk, int D,
                                                       const float* __restrict__ qscale, float cap,
                                                       const float* __restrict__ mask, float* __restrict__ out,
                                                       bf16* __restrict__ outs, int ldo) {
  __shared__ float qs[256];
  __shared__ float p[256];
  __shared__ float red[kT / 64];
  const int i = blockIdx.x, h = blockIdx.y;
  for (int d = threadIdx.x; d < D; d += kT) {
    const float qv = q[(size_t)i * ldq + h * D + d];
    qs[d] = qscale ? qv * qscale[d] : qv;
  }
  __syncthreads();
  const int j = threadIdx.x;
  float s = -INFINITY;
  if (j < Sk) {
    const float* kr = k + (size_t)j * ldk + h * D;
    float acc = 0.f;
    for (int d = 0; d < D; ++d) acc += qs[d] * kr[d];
    s = acc * (1.0f / sqrtf((float)D));
    if (cap > 0.f) s = cap * tanhf(s / cap);
    if (mask) s += mask[j];
  }
  const float m = block_max(s, red);
  const float e = j < Sk ? expf(s - m) : 0.f;
  const float sum = block_sum(e, red);
  p[j] = e / sum;
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += kT) {
    float acc = 0.f;
    for (int t = 0; t < Sk; ++t) acc += p[t] * v[(size_t)t * ldv + h * D + d];
    if (outs)
      store_split(outs, split_index(i, h * D + d, ldo), acc);
    else
      out[(size_t)i * ldo + h * D + d] = acc;
  }
}

// The same attention for a block of 4 queries of one head (self-attention of
// the text layers: Sk <= 128, D <= 64, D % 4 == 0): the head's K and V rows
// are staged in LDS (16-byte global loads) once per block instead of being
// read from global memory per query.  Wave r owns query row r: its lanes
// score keys l and l + 64 (rows padded to D + 1 floats: a half-wave's keys sit
// in distinct banks), the softmax runs in registers, and lane l < D then sums
// output column l.
constexpr int kAttQ = 4, kAttSk = 128, kAttD = 64;
__global__ __launch_bounds__(kT) void k_coca_attention_tile(const float* __restrict__ q, int ldq,
                                                            const float* __restrict__ k, int ldk,
                                                            const float* __restrict__ v, int ldv, int Sq, int Sk,
                                                            int D, float cap, const float* __restrict__ mask,
                                                            float* __restrict__ out, bf16* __restrict__ outs,
                                                            int ldo) {
  __shared__ float ks[kAttSk][kAttD + 1];
  __shared__ float vs[kAttSk][kAttD + 1];
  __shared__ float qs[kAttQ][kAttD];
  __shared__ float ps[kAttQ][kAttSk];
  const int q0 = blockIdx.x * kAttQ, h = blockIdx.y, t = threadIdx.x;
  const int nq = min(kAttQ, Sq - q0), D4 = D >> 2;
  for (int i = t; i < Sk * D4; i += kT) {
    const int j = i / D4, c = 4 * (i - j * D4);
    const float4 kv = *reinterpret_cast<const float4*>(k + (size_t)j * ldk + h * D + c);
    const float4 vv = *reinterpret_cast<const float4*>(v + (size_t)j * ldv + h * D + c);
    ks[j][c] = kv.x;
    ks[j][c + 1] = kv.y;
    ks[j][c + 2] = kv.z;
    ks[j][c + 3] = kv.w;
    vs[j][c] = vv.x;
    vs[j][c + 1] = vv.y;
    vs[j][c + 2] = vv.z;
    vs[j][c + 3] = vv.w;
  }
  for (int i = t; i < nq * D; i += kT) {
    const int r = i / D, d = i - r * D;
    qs[r][d] = q[(size_t)(q0 + r) * ldq + h * D + d];
  }
  __syncthreads();
  const int r = t >> 6, l = t & 63;
  if (r >= nq) return;  // no barrier follows
  const float scale = 1.0f / sqrtf((float)D);
  float sc[kAttSk / 64];
#pragma unroll
  for (int m = 0; m < kAttSk / 64; ++m) {
    const int j = l + 64 * m;
    float s = -INFINITY;
    if (j < Sk) {
      float acc = 0.f;
      for (int d = 0; d < D; ++d) acc += qs[r][d] * ks[j][d];
      s = acc * scale;
      if (cap > 0.f) s = cap * tanhf(s / cap);
      if (mask) s += mask[j];
    }
    sc[m] = s;
  }
  float mx = sc[0];
#pragma unroll
  for (int m = 1; m < kAttSk / 64; ++m) mx = fmaxf(mx, sc[m]);
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  float sum = 0.f;
#pragma unroll
  for (int m = 0; m < kAttSk / 64; ++m) {
    sc[m] = l + 64 * m < Sk ? expf(sc[m] - mx) : 0.f;
    sum += sc[m];
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
#pragma unroll
  for (int m = 0; m < kAttSk / 64; ++m)
    if (l + 64 * m < Sk) ps[r][l + 64 * m] = sc[m] / sum;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the row's probabilities are in LDS
  if (l < D) {
    float acc = 0.f;
    for (int j = 0; j < Sk; ++j) acc += ps[r][j] * vs[j][l];
    if (outs)
      store_split(outs, split_index(q0 + r, h * D + l, ldo), acc);
    else
      out[(size_t)(q0 + r) * ldo + h * D + l] = acc;
  }
}

// rvq.cpp:24-62, one vector: per level, every code's distance (|r|^2 - 2
// r.c) + |c|^2, the first minimum, then residual -= the chosen row.  One launch
// per level, one wave per code: every block first repeats the previous level's
// argmin over its C distances and forms the residual in LDS, so no block waits
// for another; block 0 leaves the residual and the token.  The launch after the
// last level only finishes it.  A level streams C x D floats (3.1 MB) and its
// chain is one argmin and two memory round trips; one workgroup for all levels
// (a thread per code, lanes a whole row apart) took 2,078 us for 12 x 1024 x
// 768 on MI355X.
constexpr int kRvqWaves = 4;

__global__ __launch_bounds__(64 * kRvqWaves) void k_rvq_level(const float* __restrict__ res_in,
                                                              const float* __restrict__ dist_in,
                                                              const float* __restrict__ cb_prev,
                                                              const float* __restrict__ cb, int C, int D,
                                                              float* __restrict__ res_out,
                                                              float* __restrict__ dist_out, int* __restrict__ token) {
  __shared__ float r[4096];
  __shared__ float bestv[kRvqWaves];
  __shared__ int besti[kRvqWaves];
  const int t = threadIdx.x, l = t & 63, w = t >> 6;
  if (cb_prev != nullptr) {
    // first minimum of the previous level: (value, index), the lower index on
    // ties; a NaN distance counts as infinity
    float dist = INFINITY;
    int idx = 0x7fffffff;
    for (int c = t; c < C; c += 64 * kRvqWaves) {
      float v = dist_in[c];
      v = v == v ? v : INFINITY;
      if (v < dist || (v == dist && c < idx)) {
        dist = v;
        idx = c;
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(dist, o);
      const int oi = __shfl_xor(idx, o);
      if (ov < dist || (ov == dist && oi < idx)) {
        dist = ov;
        idx = oi;
      }
    }
    if (l == 0) {
      bestv[w] = dist;
      besti[w] = idx;
    }
    __syncthreads();
    dist = bestv[0];
    idx = besti[0];
#pragma unroll
    for (int u = 1; u < kRvqWaves; ++u)
      if (bestv[u] < dist || (bestv[u] == dist && besti[u] < idx)) {
        dist = bestv[u];
        idx = besti[u];
      }
    idx = idx < C ? idx : 0;
    if (blockIdx.x == 0 && t == 0) *token = idx;
    const float* chosen = cb_prev + (size_t)idx * D;
    for (int d = t; d < D; d += 64 * kRvqWaves) {
      const float v = res_in[d] - chosen[d];
      r[d] = v;
      if (blockIdx.x == 0) res_out[d] = v;
    }
  } else {
    for (int d = t; d < D; d += 64 * kRvqWaves) r[d] = res_in[d];
  }
  __syncthreads();
  const int c = blockIdx.x * kRvqWaves + w;
  if (cb == nullptr || c >= C) return;
  const float* row = cb + (size_t)c * D;
  float r2 = 0.f, cross = 0.f, c2 = 0.f;
#pragma unroll 4
  for (int d = l; d < D; d += 64) {
    const float x = row[d], y = r[d];
    r2 += y * y;
    cross += y * x;
    c2 += x * x;
  }
  r2 = wave_sum(r2);
  cross = wave_sum(cross);
  c2 = wave_sum(c2);
  if (l == 0) dist_out[c] = (r2 - 2.0f * cross) + c2;
}

}  // namespace

void coca_embed(const int* ids, int rows, const float* table, int vocab, int D, float scale, float* x,
                hipStream_t s) {
  hipLaunchKernelGGL(k_coca_embed, dim3(rows), dim3(kT), 0, s, ids, table, vocab, D, scale, x);
  MRT_HIP_CHECK(hipGetLastError());
}

void layer_norm_rows(const float* x, int rows, int D, const float* w, const float* b, float eps, float* y, bf16* ys,
                     hipStream_t s) {
  hipLaunchKernelGGL(k_layer_norm, dim3(rows), dim3(kT), 0, s, x, D, w, b, eps, y, ys);
  MRT_HIP_CHECK(hipGetLastError());
}

void coca_attention(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv, int Sq, int Sk, int H,
                    int D, const float* qscale, float cap, const float* mask, float* out, bf16* outs, hipStream_t s) {
  MRT_REQUIRE(Sk >= 1 && Sk <= kT && D >= 1 && D <= 256, "coca attention: Sk <= 256 and d_head <= 256");
  if (!qscale && Sk <= kAttSk && D <= kAttD && D % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 &&
      reinterpret_cast<uintptr_t>(k) % 16 == 0 && reinterpret_cast<uintptr_t>(v) % 16 == 0) {
    // query blocks with the head's K / V in LDS
    hipLaunchKernelGGL(k_coca_attention_tile, dim3((Sq + kAttQ - 1) / kAttQ, H), dim3(kT), 0, s, q, ldq, k, ldk, v,
                       ldv, Sq, Sk, D, cap, mask, out, outs, H * D);
  } else {
    hipLaunchKernelGGL(k_coca_attention, dim3(Sq, H), dim3(kT), 0, s, q, ldq, k, ldk, v, ldv, Sk, D, qscale, cap,
                       mask, out, outs, H * D);
  }
  MRT_HIP_CHECK(hipGetLastError());
}

void rvq_quantize(const float* vec, const float* codebooks, int K, int C, int D, float* work, float* residual,
                  int* tokens, hipStream_t s) {
  MRT_REQUIRE(K >= 1 && C >= 1 && C <= 1024 && D >= 1 && D <= 4096, "rvq_quantize: codebook <= 1024, dim <= 4096");
  // two residuals and two rows of distances, alternating by level
  float* res[2] = {work, work + D};
  float* dist[2] = {work + 2 * D, work + 2 * D + C};
  const size_t level = static_cast<size_t>(C) * D;
  for (int k = 0; k <= K; ++k) {
    const bool last = k == K;
    const float* res_in = k <= 1 ? vec : res[(k - 1) & 1];  // the residual entering level k - 1 (level 0: vec)
    hipLaunchKernelGGL(k_rvq_level, dim3(last ? 1 : (C + kRvqWaves - 1) / kRvqWaves), dim3(64 * kRvqWaves), 0, s,
                       res_in, dist[(k - 1) & 1], k > 0 ? codebooks + (k - 1) * level : nullptr,
                       last ? nullptr : codebooks + k * level, C, D, last ? residual : res[k & 1], dist[k & 1],
                       tokens + (k > 0 ? k - 1 : 0));
    MRT_HIP_CHECK(hipGetLastError());
  }
}

}  // namespace mrt
