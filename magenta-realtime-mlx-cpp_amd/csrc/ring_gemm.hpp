// The multiply loop of the matrix-core GEMMs: BM x BN tiles, WM x WN waves, k-tiles
// streamed global -> LDS through a ring of S stages.
//
// A wave keeps two fragment sets: the fragments of a 16-deep step are read from
// LDS between the products of the step before it, also across the barrier to the
// next k-tile, so LDS reads and matrix instructions of one wave overlap (all
// reads of a k-tile ahead of its products: 818 us, 908 TFLOP/s, at 64,384 x 5,632 x
// 1,024 in cache, two 192 x 128 blocks a CU; this loop 666 us).  The products are taken as B A^T, so a lane's
// accumulators lie along one output row and the epilogue stores 16 bytes a lane.
#pragma once

#include "mfma_ring.hpp"

namespace mrt {

typedef float f32x8_t __attribute__((ext_vector_type(8)));

// The 32x32x16 matrix instruction of each 16-bit storage type (fp32 accumulators).
// Operand fragments: lane l holds row (l % 32) and k = 8 (l / 32) .. + 7 of both
// operands; accumulator r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4 of the
// first operand against row l % 32 of the second.
template <typename T>
struct Mfma;
template <>
struct Mfma<bf16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  __device__ __forceinline__ static f32x16_t mma(v8 a, v8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<f16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  __device__ __forceinline__ static f32x16_t mma(v8 a, v8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// 16-bit operands: a k-tile is 64 deep, a row of it 8 chunks of 16 bytes; chunk c of
// row r is stored at chunk c ^ swz(r), so the 32 rows x 2 chunks of a fragment read
// (and 16 consecutive lanes of any ds_read_b128) fall in distinct banks.
template <typename T>
struct Core16 {
  typedef typename Mfma<T>::v8 v8;
  static constexpr int kChunks = 8, kSteps = 4, kParts = 1, kDepth = 64;
  __device__ static int swz(int r) { return (r ^ (r >> 3)) & 7; }
  __device__ static int place(int r, int chunk) { return chunk ^ swz(r); }
  __device__ static int chunk_at(int r, int pos) { return pos ^ swz(r); }
  __device__ static int chunk(int step, int, int half) { return 2 * step + half; }
  __device__ __forceinline__ static void mma(const v8 (&a)[1], const v8 (&b)[1], int, f32x16_t& c) {
    c = Mfma<T>::mma(b[0], a[0], c);
  }
  static constexpr int kProducts = 1;
  static constexpr bool kFine = false;
};

template <class Core, int BM, int BN, int WM, int WN, int S>
struct RingTile {
  typedef typename Core::v8 v8;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves, kBM = BM, kBN = BN, kS = S;
  static constexpr int MI = BM / WM / 32, NJ = BN / WN / 32;  // 32 x 32 tiles of a wave
  static constexpr int kRow = Core::kChunks * 16;             // bytes of a row of a k-tile
  static constexpr int kStage = (BM + BN) * kRow;
  static constexpr int LA = BM * Core::kChunks / kThreads, LB = BN * Core::kChunks / kThreads;  // loads of a thread
  static constexpr size_t kLds = (size_t)S * kStage;
  static_assert(BM * Core::kChunks % kThreads == 0 && BN * Core::kChunks % kThreads == 0, "whole loads per wave");
  static_assert(BM % (32 * WM) == 0 && BN % (32 * WN) == 0, "whole 32 x 32 tiles per wave");
  static_assert(kLds <= 160 * 1024 && (S - 1) * (LA + LB) < 64, "LDS of one CU, vmcnt range");

  // row and source chunk of load q of this thread
  __device__ static void load_pos(int q, int& row, int& chunk) {
    const int idx = (q * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 64 + (threadIdx.x & 63);
    row = idx / Core::kChunks;
    chunk = Core::chunk_at(row, idx - row * Core::kChunks);
  }
  __device__ static void load_a(unsigned char* stage, int q, const void* src) { load(stage, q, src); }
  __device__ static void load_b(unsigned char* stage, int q, const void* src) { load(stage + BM * kRow, q, src); }

  struct State {
    f32x16_t acc[MI][NJ];  // (i, j), r: row 32 i + lane % 32, column 32 j + 8 (r / 4) + 4 (lane / 32) + r % 4
    f32x16_t low[Core::kFine ? MI : 1][Core::kFine ? NJ : 1];  // sums of all products but the last
    v8 a[2][MI][Core::kParts], b[2][NJ][Core::kParts];
    int slot = 0;  // ring stage of the next k-tile
    __device__ void clear() {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            acc[i][j][r] = 0.f;
            if constexpr (Core::kFine) low[i][j][r] = 0.f;
          }
    }
    // acc the whole sums
    __device__ void settle() {
      if constexpr (Core::kFine) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[i][j] += low[i][j];
      }
    }
  };

  // Fill the ring (issue(stage) requests the next k-tile of the stream) and read
  // the first fragments.
  template <class Issue>
  __device__ static void start(unsigned char* lds, State& s, Issue&& issue) {
#pragma unroll
    for (int t = 0; t < S; ++t) issue(lds + t * kStage);
    __builtin_amdgcn_s_waitcnt(vm_wait_imm((S - 1) * (LA + LB)));
    ring_barrier();
    read(lds, 0, 0, s);
  }

  // Multiply one k-tile.  wait() returns once this wave's loads of the next
  // k-tile have landed: all but the S - 2 k-tiles requested after it
  // (wait_loads), plus what else the wave has issued since.
  template <class Issue, class Wait>
  __device__ static void ktile(unsigned char* lds, State& s, Issue&& issue, Wait&& wait) {
    unsigned char* st = lds + s.slot * kStage;
    s.slot = s.slot + 1 == S ? 0 : s.slot + 1;
#pragma unroll
    for (int t = 0; t + 1 < Core::kSteps; ++t) {
      read(st, t + 1, (t + 1) & 1, s);
      products(t & 1, s);
      interleave();
    }
    wait();
    ring_barrier();  // every wave's loads of the next k-tile; every wave has read this one
    issue(st);
    read(lds + s.slot * kStage, 0, 0, s);
    products((Core::kSteps - 1) & 1, s);
    interleave();
  }

  // The first fragments of the next k-tile again.
  __device__ static void reread(unsigned char* lds, State& s) { read(lds + s.slot * kStage, 0, 0, s); }

  // Row and column of sum e (acc[e / 16 / NJ][e / 16 % NJ], r = e % 16) in the tile.
  __device__ static void sum_pos(int e, int& row, int& col) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = e / 16 / NJ, j = e / 16 % NJ, r = e % 16;
    row = (wid / WN) * (BM / WM) + 32 * i + (lane & 31);
    col = (wid % WN) * (BN / WN) + 32 * j + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
  }

  // Extra: vector memory instructions issued after the loads waited for.
  template <int Extra = 0>
  __device__ static void wait_loads() {
    constexpr int n = (S - 2) * (LA + LB) + Extra;
    __builtin_amdgcn_s_waitcnt(vm_wait_imm(n < 63 ? n : 63));
  }

 private:
  __device__ static void load(unsigned char* dst, int q, const void* src) {
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __builtin_amdgcn_global_load_lds((const MRT_GLOBAL void*)src, (MRT_LDS void*)(dst + (q * kWaves + wid) * 1024), 16,
                                     0, 0);
  }
  __device__ static void read(const unsigned char* st, int step, int d, State& s) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 31, lh = lane >> 5;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int r = (wid / WN) * (BM / WM) + i * 32 + lr;
#pragma unroll
      for (int p = 0; p < Core::kParts; ++p)
        s.a[d][i][p] = *reinterpret_cast<const v8*>(st + r * kRow + Core::place(r, Core::chunk(step, p, lh)) * 16);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = (wid % WN) * (BN / WN) + j * 32 + lr;
#pragma unroll
      for (int p = 0; p < Core::kParts; ++p)
        s.b[d][j][p] =
            *reinterpret_cast<const v8*>(st + BM * kRow + r * kRow + Core::place(r, Core::chunk(step, p, lh)) * 16);
    }
  }
  __device__ static void products(int d, State& s) {
#pragma unroll
    for (int u = 0; u < Core::kProducts; ++u)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          if constexpr (Core::kFine)
            Core::mma(s.a[d][i], s.b[d][j], u, u + 1 < Core::kProducts ? s.low[i][j] : s.acc[i][j]);
          else
            Core::mma(s.a[d][i], s.b[d][j], u, s.acc[i][j]);
        }
  }
  // One product, then its share of the next step's LDS reads.
  __device__ static void interleave() {
    constexpr int kReads = (MI + NJ) * Core::kParts, kMfma = MI * NJ * Core::kProducts;
#pragma unroll
    for (int r = 0; r < kMfma; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, (kReads + kMfma - 1) / kMfma, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
};

}  // namespace mrt
