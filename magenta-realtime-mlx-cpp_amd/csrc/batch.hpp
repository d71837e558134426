// Batched independent streams: B streams (each its own encoder tokens, seed,
// KV caches) decoded together as R = 2B activation rows, so every projection
// is one skinny GEMM on the matrix cores and the weights stream once per step
// for all streams.  Per stream the semantics are those of generate_tokens
// (depthformer/decode.cpp:239-573) at batch 1.
#pragma once

#include <cstdint>
#include <vector>

#include "common.hpp"
#include "model.hpp"

namespace mrt {

constexpr int kBatchRows = 64;  // activation rows of one batched step (32 streams)

// Fragment order: the operands of the skinny GEMMs are stored as 16-row x
// 32-column tiles, each tile the 64 lanes' 16-byte operands of one 16x16x32
// matrix instruction (lane l: row l % 16, columns 8 (l / 16) .. + 7), tiles of a
// row group back to back along K.  Element (m, k): frag_index (device_utils.hpp).
// Activation buffers hold whole tiles: frag_rows(M) rows.
inline int frag_rows(int M) { return (M + 15) / 16 * 16; }

// Elements of an (N, K) weight matrix in fragment order (N padded to 16 rows,
// and 16 rows more).
size_t frag_weights_elems(int N, int K);
// The matrix in fragment order.  pairs: W is a packed wi_0 / wi_1 matrix (N = 2F
// rows, bgemm_geglu).
void frag_weights(DType dt, const void* W, int N, int K, bool pairs, void* out, hipStream_t s);

// RMSNorm (eps, weights g) of a GEMM's input rows applied between their load and
// the products: X then holds the raw residual rows, whose sums of squares are
// the K / 16 partials per row that the bgemm_resid which last wrote them left at
// ssq.  g == nullptr: X is used as it is.
struct BNorm {
  const void* g = nullptr;
  const float* ssq = nullptr;
  float eps = 0.f;
};

// Skinny GEMMs Y (M x N) = X (M x K) . W^T, 16-bit storage types, fp32
// accumulation, M <= 64, K % 32 == 0, X and W in fragment order
// (batch_kernels.hip).  Epilogues as the batch-1 GEMVs.
void bgemm_store(DType dt, const void* X, int M, int K, const void* W, int N, void* Y, int ldy, hipStream_t s,
                 const BNorm& norm = {});
// Logits, rounded to the storage type: weight rows w_row0 .. + N.  groups > 1:
// independent products, rows [g M, + M) of X against weight rows
// w_row0 + g w_group_rows .. + N into Y rows g M + m.
void bgemm_f32(DType dt, const void* X, int M, int K, const void* W, int w_row0, int N, float* Y, int ldy,
               hipStream_t s, const BNorm& norm = {}, int groups = 1, int w_group_rows = 0);
// R (M, N) += X . W^T (rounded as the batch-1 residual); the updated rows also
// in fragment order to Rf, and each row's sums of squares over its 16-column
// tiles to ssq (M, N / 16).
void bgemm_resid(DType dt, const void* X, int M, int K, const void* W, int N, void* R, void* Rf, float* ssq,
                 hipStream_t s);
// W = [Wq; Wk; Wv] (3 HD rows): q -> Q (M, HD); k, v -> ring slot pos (or
// *pos_ptr when non-null) of caches laid out (M, H, Lmax, 64).
void bgemm_qkv(DType dt, const void* X, int M, int K, const void* W, int HD, void* Q, void* Kc, void* Vc, int H,
               int Lmax, int pos, const int* pos_ptr, hipStream_t s, const BNorm& norm = {});
// The same for rows m = P * pos + r (positions of one stream's frame, P CFG
// rows each): k / v -> slot pos of ring row r (P, H, Lmax, 64).
void bgemm_qkv_pos(DType dt, const void* X, int M, int K, const void* W, int HD, void* Q, void* Kc, void* Vc, int H,
                   int Lmax, int P, hipStream_t s);
// Gated GELU over the 32-row packed wi_0 / wi_1 matrix (2F rows) -> (M, F) in
// fragment order.
void bgemm_geglu(DType dt, const void* X, int M, int K, const void* W01, int F, void* Hout, hipStream_t s,
                 const BNorm& norm = {});

// The same products with every output summed over k in order, bit for bit as gemm()
// sums them (any M): row-major Y (M, N), fp32 logits, R += X . W^T, and gated GELU
// in fragment order.
void bgemm_seq_store(DType dt, const void* X, int M, int K, const void* W, int N, void* Y, hipStream_t s);
void bgemm_seq_f32(DType dt, const void* X, int M, int K, const void* W, int N, float* Y, hipStream_t s);
void bgemm_seq_resid(DType dt, const void* X, int M, int K, const void* W, int N, void* R, hipStream_t s);
void bgemm_seq_geglu(DType dt, const void* X, int M, int K, const void* W01, int F, void* Hout, hipStream_t s);

// Cross attention (no bias, no mask, scale 1) of every (row, head) over S <=
// 1024 encoder keys, caches laid out (rows, H, S, 64); out (rows, H * 64) in
// fragment order.
void cross_attn_rows(const void* Q, const void* Kc, const void* Vc, int rows, int H, int S, void* out, hipStream_t s);

// Gumbel noise of every draw for every stream: out (streams, frames, L, C).
void gumbel_tables(const uint64_t* seeds, int streams, int frames, int L, int C, float* out, hipStream_t s);

// Device frame counter of a replayed frame graph.
void set_counter(int* p, int v, hipStream_t s);
void advance_counter(int* p, hipStream_t s);

class Batch {
 public:
  Batch(Model& m, int streams, int max_frames, int enc_len);
  ~Batch();
  Batch(const Batch&) = delete;
  Batch& operator=(const Batch&) = delete;

  Model& m;
  int B, R, F, S;
  hipStream_t stream = nullptr;

  // tokens: host (R, S); rows 2b and 2b + 1 are stream b's CFG pair.
  void encode(const int32_t* tokens_host);
  void encode_device();
  int* enc_tokens_dev() const { return enc_.tok; }
  // One chunk of every stream.  seeds: host (B); o.teacher: host (B, F, L)
  // or null; out: host (B, num_frames, L) LLM ids.  o.record_slices (device
  // (F, L, R, C)) and o.record_temporal (device (F, R, D)) run the loop
  // without the frame graph.
  void generate(const int32_t* enc_tokens_host, const GenOpts& o, const uint64_t* seeds, int32_t* out_host);
  // GPU ms of the last generate call's decode section.
  float last_decode_ms() const;
  void* enc_out() const { return enc_.enc_out; }

 private:
  void enqueue_frame(const GenOpts& o, int f, bool dynamic);
  void temporal_stack(int f, const int* fptr);
  void depth_stack(void* x, int l, bool x_partials, bool qkv_fed);
  // the norm (weights g) of a GEMM input whose row partials are at ssq_
  BNorm norm(const void* g) const { return BNorm{g, ssq_, 1e-6f}; }
  void* dalloc(size_t bytes);
  void setup();
  void release();
  char* ring(void* base, int layer, int kv, int len) const;

  std::vector<void*> allocs_;
  EncoderBufs enc_;
  bool encoded_ = false;
  void *tkv_ = nullptr, *dkv_ = nullptr;
  void *t_in_ = nullptr, *d_in_ = nullptr, *xn_ = nullptr, *q_ = nullptr, *att_ = nullptr, *ffh_ = nullptr;
  // the last residual update: its rows in fragment order and their partials (R, d_model / 16)
  void* xf_ = nullptr;
  float* ssq_ = nullptr;
  const std::vector<FragLayer>* tmp_ = nullptr;  // the model's
  const FragDepth* dep_ = nullptr;
  // the model's depth layer-0 q/k/v table of the current call's codec levels,
  // or nullptr (layer 0 computed at every level)
  const void* qkv_tab_ = nullptr;
  void* fsum_ = nullptr;
  float* logits_ = nullptr;
  float* noise_ = nullptr;  // (B, F, L, 1024) Gumbel noise of the current call
  int *d_tokens_ = nullptr, *d_teacher_ = nullptr, *d_frame_ = nullptr;
  uint64_t* d_seeds_ = nullptr;
  int32_t* h_pinned_ = nullptr;
  size_t h_pinned_n_ = 0;
  hipEvent_t ev_[2] = {nullptr, nullptr};
  bool timed_ = false;
  hipGraph_t graph_ = nullptr;
  hipGraphExec_t graph_exec_ = nullptr;
  std::vector<double> graph_key_;
};

}  // namespace mrt
