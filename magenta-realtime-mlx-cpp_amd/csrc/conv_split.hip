// fp32 convolutions (and one-tap GEMMs) on the bf16 matrix cores: implicit GEMM on
// split operands (split_gemm.hpp) through the ring of ring_gemm.hpp.
//
// Rows of the first operand are output pixels: k-tile (tap, 32 channels) of a pixel
// is one 192-byte group of the input pixel under that tap, loaded straight into
// LDS, or a group of zeros outside the input.  Rows of the second are output
// channels, their weights laid out as split rows of taps x cin values.  The
// producers write split activations, with the ELU applied where the consumer wants
// it.  Against k_conv (fp32 matrix instruction, operands through registers) the
// codec's 51 frames take 3.21 -> 2.21 ms (MI355X; with the output conv 117 -> 91 us), error
// against 64 bits 2.1e-6 -> 1.4e-6.
#include <algorithm>
#include <type_traits>

#include "codec.hpp"
#include "split_gemm.hpp"

namespace mrt {
namespace {

__device__ __forceinline__ float elu1(float v) { return v > 0.f ? v : expf(v) - 1.f; }

// The epilogue of one output pixel's channels o .. o + 3: bias, residual,
// activation, fp32 and split stores.
struct PixelOut {
  size_t row, res;  // output pixel (of stereo half 0), residual pixel
  size_t half;      // pixels from one stereo half to the next
};

__device__ __forceinline__ PixelOut pixel_out(const ConvLaunch& a, const ConvSub* sub, int m) {
  const int gy = sub->gy, gx = sub->gx;
  const int img = m / (gy * gx), r = m - img * gy * gx;
  const int yy = r / gx, xx = r - yy * gx;
  const int oy = yy * sub->oys + sub->oyo, ox = xx * sub->oxs + sub->oxo;
  PixelOut p;
  p.row = ((size_t)img * a.hout + oy) * a.wout + ox;
  p.half = (size_t)a.n * a.hout * a.wout;
  p.res = a.res ? ((size_t)img * a.res_h + oy / a.rh) * a.res_w + ox / a.rw : 0;
  return p;
}

__device__ __forceinline__ void conv_store4(const ConvLaunch& a, const PixelOut& p, int o, float (&v)[4]) {
  if (a.bias) {
    const float4 b = *reinterpret_cast<const float4*>(a.bias + o);
    v[0] += b.x, v[1] += b.y, v[2] += b.z, v[3] += b.w;
  }
  if (a.res) {
    const float4 b = *reinterpret_cast<const float4*>(a.res + p.res * a.cout + o);
    v[0] += b.x, v[1] += b.y, v[2] += b.z, v[3] += b.w;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (a.act_out == kActElu) v[e] = elu1(v[e]);
    if (a.act_out == kActGelu) v[e] = v[e] * 0.5f * (1.0f + erff(v[e] * 0.7071067811865475f));
  }
  const int h = o >= a.split ? o / a.split : 0, oc = o - h * a.split;
  const size_t row = p.row + h * p.half;
  if (a.y) *reinterpret_cast<float4*>(a.y + row * a.split + oc) = make_float4(v[0], v[1], v[2], v[3]);
  if (a.ys) store_split4(a.ys, split_index(row, oc, a.split), v);
  if (!a.y_elu && !a.ys_elu) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = elu1(v[e]);
  if (a.y_elu) *reinterpret_cast<float4*>(a.y_elu + row * a.split + oc) = make_float4(v[0], v[1], v[2], v[3]);
  if (a.ys_elu) store_split4(a.ys_elu, split_index(row, oc, a.split), v);
}

// Small tiles take long sums (the large ones are chosen for many pixels) and keep
// their small products apart: the style model's error against 64 bits is 1.2e-6
// without, 0.97e-6 with (fp32 matrix instruction: 1.1e-6), at the same time.
template <int BM, int BN, int WM, int WN, int S>
using ConvTile = RingTile<std::conditional_t<BM * BN <= 128 * 64, CoreSplitFine, CoreSplit>, BM, BN, WM, WN, S>;

// Block (x, y, z): pixel tile x, channel tile y, slice z of the k-tiles.  Slices of
// one tile leave their sums in `partial` and count themselves in counters[tile];
// the one that comes last adds all slices in order, so the result does not depend
// on which it is, and no block waits.  Partial sums are stored and read at agent
// scope (through the XCDs' L2s), and a block's have reached memory (vmcnt 0 in
// every wave, then the barrier) before it counts itself.
template <int BM, int BN, int WM, int WN, int S, int MINW>
__global__ __launch_bounds__(64 * WM * WN, MINW) void k_conv_split(ConvLaunch a) {
  using Tile = ConvTile<BM, BN, WM, WN, S>;
  extern __shared__ __align__(16) unsigned char lds[];
  int si = 0;
  while (si + 1 < a.nsub && (int)blockIdx.x >= a.subs[si + 1].tile0) ++si;
  const ConvSub* sub = a.subs + si;
  const int gx = sub->gx, gyx = sub->gy * gx, M = a.n * gyx;
  const int m0 = ((int)blockIdx.x - sub->tile0) * BM, n0 = (int)blockIdx.y * BN;
  const int cpt = a.cin >> 5, nk_all = sub->ntaps * cpt;
  const int kb = (int)((long)blockIdx.z * nk_all / a.ksplit), ke = (int)((long)(blockIdx.z + 1) * nk_all / a.ksplit);

  // this thread's rows: linear input pixel, grid coordinates, chunk
  int lin[Tile::LA], py[Tile::LA], px[Tile::LA], ac[Tile::LA];
  const bf16 *ap[Tile::LA], *bp[Tile::LB];
#pragma unroll
  for (int q = 0; q < Tile::LA; ++q) {
    int row, chunk;
    Tile::load_pos(q, row, chunk);
    const int m = min(m0 + row, M - 1), img = m / gyx, r = m - img * gyx;
    py[q] = r / gx;
    px[q] = r - py[q] * gx;
    lin[q] = (img * a.hin + py[q]) * a.win + px[q];
    ac[q] = chunk * 8;
  }
#pragma unroll
  for (int q = 0; q < Tile::LB; ++q) {
    int row, chunk;
    Tile::load_pos(q, row, chunk);
    bp[q] = static_cast<const bf16*>(sub->w) + ((size_t)(n0 + row) * nk_all + kb) * kSplitGroup + chunk * 8;
  }
  int kt = kb, tap = kb / cpt, grp = kb - tap * cpt;
  auto point = [&]() {  // the input pixels under tap `tap`, channel group `grp`
    const int dy = sub->dy[tap], dx = sub->dx[tap], d = dy * a.win + dx;
#pragma unroll
    for (int q = 0; q < Tile::LA; ++q) {
      const bool in = (unsigned)(py[q] + dy) < (unsigned)a.hin && (unsigned)(px[q] + dx) < (unsigned)a.win;
      const bf16* base = in ? a.xs + (size_t)(lin[q] + d) * (cpt * kSplitGroup) : a.zeros;
      ap[q] = base + grp * kSplitGroup + ac[q];
    }
  };
  point();
  auto issue = [&](unsigned char* stage) {
#pragma unroll
    for (int q = 0; q < Tile::LA; ++q) Tile::load_a(stage, q, ap[q]);
#pragma unroll
    for (int q = 0; q < Tile::LB; ++q) Tile::load_b(stage, q, bp[q]);
    if (kt + 1 < ke) {  // past the end: the last k-tile again, into a free stage
      ++kt;
#pragma unroll
      for (int q = 0; q < Tile::LB; ++q) bp[q] += kSplitGroup;
      if (++grp == cpt) {
        grp = 0;
        ++tap;
        point();
      } else {
#pragma unroll
        for (int q = 0; q < Tile::LA; ++q) ap[q] += kSplitGroup;
      }
    }
  };

  typename Tile::State s;
  Tile::start(lds, s, issue);
  s.clear();
  for (int k = kb; k < ke; ++k) Tile::ktile(lds, s, issue, [] { Tile::template wait_loads<>(); });
  s.settle();
  __builtin_amdgcn_s_waitcnt(vm_wait_imm(0));  // no copy into LDS outlives the block

  if (a.ksplit > 1) {
    typedef unsigned long long u64;
    constexpr int kQuads = Tile::MI * Tile::NJ * 4;  // per thread
    const unsigned tile = blockIdx.x * gridDim.y + blockIdx.y;
    u64* part = reinterpret_cast<u64*>(a.partial) + (size_t)tile * a.ksplit * (BM * BN / 2) + threadIdx.x;
    u64* mine = part + (size_t)blockIdx.z * (BM * BN / 2);
#pragma unroll
    for (int q = 0; q < kQuads; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x16_t& c = s.acc[q / 4 / Tile::NJ][q / 4 % Tile::NJ];
        const u64 w = (u64)__float_as_uint(c[4 * (q & 3) + 2 * h]) |
                      ((u64)__float_as_uint(c[4 * (q & 3) + 2 * h + 1]) << 32);
        __hip_atomic_store(mine + (2 * q + h) * Tile::kThreads, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    unsigned* last = reinterpret_cast<unsigned*>(lds);
    __syncthreads();
    if (threadIdx.x == 0) {
      const unsigned old =
          __hip_atomic_fetch_add(a.counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = old + 1 == (unsigned)a.ksplit;
      if (old + 1 == (unsigned)a.ksplit)  // ready for the next launch
        __hip_atomic_store(a.counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*last) return;
    s.clear();
    for (int z = 0; z < a.ksplit; ++z) {
      const u64* src = part + (size_t)z * (BM * BN / 2);
#pragma unroll
      for (int q = 0; q < kQuads; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const u64 w = __hip_atomic_load(src + (2 * q + h) * Tile::kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          f32x16_t& c = s.acc[q / 4 / Tile::NJ][q / 4 % Tile::NJ];
          c[4 * (q & 3) + 2 * h] += __uint_as_float((unsigned)w);
          c[4 * (q & 3) + 2 * h + 1] += __uint_as_float((unsigned)(w >> 32));
        }
    }
  }
  resum_not_finite<Tile>(s, [&](int row, int col) {
    const int m = min(m0 + row, M - 1), img = m / gyx, r = m - img * gyx, y = r / gx, x = r - y * gx;
    const bf16* w = static_cast<const bf16*>(sub->w) + (size_t)(n0 + col) * nk_all * kSplitGroup;
    float sum = 0.f;
    for (int t = 0; t < sub->ntaps && sum == sum; ++t, w += cpt * kSplitGroup) {
      const int iy = y + sub->dy[t], ix = x + sub->dx[t];
      const bool in = (unsigned)iy < (unsigned)a.hin && (unsigned)ix < (unsigned)a.win;
      sum = split_dot(in ? a.xs + ((size_t)(img * a.hin + iy) * a.win + ix) * (cpt * kSplitGroup) : a.zeros, w, cpt,
                      sum);
    }
    return sum;
  });
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < Tile::MI; ++i) {
    const int m = m0 + (wid / WN) * (BM / WM) + 32 * i + (lane & 31);
    if (m >= M) continue;
    const PixelOut p = pixel_out(a, sub, m);
#pragma unroll
    for (int j = 0; j < Tile::NJ; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int o = n0 + (wid % WN) * (BN / WN) + 32 * j + 8 * g + 4 * (lane >> 5);
        if (o >= a.cout) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = s.acc[i][j][4 * g + e];
        conv_store4(a, p, o, v);
      }
  }
}

// The tiles, with their measured costs (us): a k-tile in a block that has a CU to
// itself and in one of two on a CU, and a round's ring fill and epilogue.
struct TileInfo {
  int bm, bn, per_cu;
  double alone, shared, round;
};
constexpr TileInfo kTiles[] = {{256, 128, 1, 2.01, 2.01, 9.5},
                               {128, 128, 1, 1.00, 1.00, 7.3},
                               {128, 64, 2, 0.70, 1.42, 5.1},
                               {64, 64, 2, 0.37, 0.84, 2.4}};

template <int BM, int BN, int WM, int WN, int S, int MINW>
void launch(const ConvLaunch& a, int tiles_m, hipStream_t s) {
  using Tile = ConvTile<BM, BN, WM, WN, S>;
  const auto kernel = &k_conv_split<BM, BN, WM, WN, S, MINW>;
  allow_dynamic_lds(reinterpret_cast<const void*>(kernel), Tile::kLds);
  hipLaunchKernelGGL(kernel, dim3(tiles_m, a.cout_pad / BN, a.ksplit), dim3(Tile::kThreads), Tile::kLds, s, a);
}

}  // namespace

// The tile and K split of least estimated time: rounds over the CUs x (k-tiles of a
// slice + round cost) + the partial sums of a split (every slice's store, the last
// slice's loads).  The constants are a least-squares fit over 17 shapes of 30 to
// 199,680 pixels, 64 to 2,560 channels, 18 to 288 k-tiles and 1 to 16 slices, and
// give their times within 8 %.
void conv_split_plan(ConvLaunch& a, const ConvSub* subs, int nsub) {
  const long cus = device_cus();
  double best = 1e30;
  for (int t = 0; t < (int)(sizeof(kTiles) / sizeof(kTiles[0])); ++t) {
    const TileInfo& T = kTiles[t];
    if (a.cout_pad % T.bn) continue;
    long tiles = 0;
    int nk = 0, min_nk = 1 << 30;
    for (int i = 0; i < nsub; ++i) {
      tiles += ((long)a.n * subs[i].gy * subs[i].gx + T.bm - 1) / T.bm;
      nk = std::max(nk, subs[i].ntaps * (a.cin / 32));
      min_nk = std::min(min_nk, subs[i].ntaps * (a.cin / 32));
    }
    tiles *= a.cout_pad / T.bn;
    for (int z = 1; z <= std::min(16, std::max(1, min_nk / 2)); ++z) {
      const long blocks = tiles * z, slots = cus * T.per_cu, rem = blocks % slots;
      const double kt = (nk + z - 1) / z, area = (double)T.bm * T.bn;
      double us = (double)(blocks / slots) * (kt * T.shared + T.round);
      if (rem) us += kt * (rem > cus ? T.shared : T.alone) + T.round;
      if (z > 1) us += 1.8 + z * area * 6.8e-5 + (double)blocks * area * 3.2e-7;
      if (us < best) {
        best = us;
        a.tile = t;
        a.ksplit = z;
      }
    }
  }
}

int conv_split_tile_rows(const ConvLaunch& a) { return kTiles[a.tile].bm; }

size_t conv_split_partial(const ConvLaunch& a, int tiles_m) {
  return a.ksplit > 1 ? (size_t)a.ksplit * tiles_m * kTiles[a.tile].bm * a.cout_pad : 0;
}
size_t conv_split_counters(const ConvLaunch& a, int tiles_m) {
  return (size_t)tiles_m * (a.cout_pad / kTiles[a.tile].bn);
}

void conv_split_launch(const ConvLaunch& a, int tiles_m, hipStream_t s) {
  switch (a.tile) {
    case 0: launch<256, 128, 4, 2, 2, 2>(a, tiles_m, s); break;
    case 1: launch<128, 128, 4, 2, 3, 2>(a, tiles_m, s); break;
    case 2: launch<128, 64, 2, 2, 2, 2>(a, tiles_m, s); break;
    default: launch<64, 64, 2, 2, 3, 2>(a, tiles_m, s); break;
  }
  MRT_HIP_CHECK(hipGetLastError());
}

}  // namespace mrt
