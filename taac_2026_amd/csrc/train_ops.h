// Internal entry points of the training stack (train.hip): the forward and backward kernels over a COMPACT tensor - the valid
// tokens of the batch, one behind the other - whose number of rows is known on the device only (count; M is an upper bound that
// sizes buffers and grids). Rows are contiguous ([M, width]) unless a stride is given; 16-byte alignment and the supported shapes
// are the caller's business (train.hip checks them once).
#pragma once

#include "common.h"

namespace taac {

// Panel order of a tall [M, N] matrix that one kernel writes and the next ones read in column slabs: panels of 256 rows x 32
// columns, each contiguous, the panels of a row block one behind the other (N and the row capacity are multiples of 32 and 256).
// A 32-column slab of 256 rows is 16 KB in one run; in row-major order it is 64-byte runs a power of two apart, which take half a
// cache line each and crowd the same memory channels.
constexpr int kPanelRows = 256, kPanelCols = 32;
constexpr int64_t kPanel = kPanelRows * kPanelCols;
inline int64_t panel_rows(int64_t M) { return (M + kPanelRows - 1) / kPanelRows * kPanelRows; }
__device__ __forceinline__ int64_t panel_row(int64_t m, int64_t N) {  // element offset of column 0 of row m
  return (m / kPanelRows) * kPanelRows * N + (m % kPanelRows) * kPanelCols;
}

// out = linear([rmsnorm](x)), K = D in {128, 256}; the norm's weight is folded into `packed` (norm_weight only says that there is
// one); rstd_out [M]: the norm's factor per row, or null.
int norm_linear_count(const char* name, const void* x, const void* norm_weight, float eps, const void* bias, const void* packed,
                      void* out, int64_t M, int32_t N, int32_t K, const int32_t* count, float* rstd_out, hipStream_t s);
// x1 = residual + linear(attn), out = x1 + feed-forward(rmsnorm(x1)); x1 and the norm's factor are kept in x1_out / rstd_out.
int attn_out_ffn_count(const char* name, const void* attn, const void* out_bias, const void* packed_out, const void* residual,
                       const void* norm_weight, float eps, const void* b_up, const void* b_down, const void* packed_ffn,
                       void* out, void* x1_out, float* rstd_out, int64_t M, int32_t D, int32_t F, bool gate_first,
                       bool act_folded, const int32_t* count, const void* head_w, float* token_dots, void* split_scratch,
                       hipStream_t s);
// Attention over samples that start at row row_offsets[b] and hold lengths[b] tokens (at most T); q | k side by side in rows of
// ld_qk elements, v in rows of ld_v, heads of dh features; lse [B, H, T]. struct_bits: visibility per sample ([T, ceil(T / 32)]
// words, struct_stride words apart) or null.
int attention_compact_fwd(const char* name, const void* qk, const void* v, int64_t ld_qk, int64_t ld_v, const int32_t* lengths,
                          const int32_t* row_offsets, const uint32_t* struct_bits, int64_t struct_stride, void* o, int64_t ld_o,
                          float* lse, int32_t B, int32_t H, int32_t T, int32_t dh, hipStream_t s);
// Its backward: dqkv = dq | dk | dv side by side in rows of ld_dqkv elements; delta [B, H, T] scratch.
int attention_compact_bwd(const char* name, const void* qk, const void* v, int64_t ld_qk, int64_t ld_v, const void* o, int64_t ld_o,
                          const void* dout, int64_t ld_do, const float* lse, const int32_t* lengths, const int32_t* row_offsets,
                          const uint32_t* struct_bits, int64_t struct_stride, void* dqkv, int64_t ld_dqkv, float* delta, int32_t B,
                          int32_t H, int32_t T, int32_t dh, hipStream_t s);
// hidden [M, F] and the gradient of the up projection [M, 2F] from x (in front of the norm; rstd its factor, norm_w [D] its weight)
// and the gradient dy of the feed-forward output. Both results are in panel order.
int ffn_bwd_hidden_count(const char* name, const void* x, const float* rstd, const void* norm_w, const void* dy, const void* packed,
                         const void* b_up, void* hidden, void* grad_pre, int64_t M, int32_t D, int32_t F, bool gate_first,
                         const int32_t* count, hipStream_t s);

// Element (row d, column c) of a weight transposed to [D, K], in the order in which dgrad_norm reads it: panels of 32 columns, D rows
// of 64 bytes each, one behind the other.
__host__ __device__ inline int64_t transposed_weight_at(int64_t d, int64_t c, int64_t D) { return c / 32 * (D * 32) + d * 32 + c % 32; }

// dx = dres + d rmsnorm(x) applied to dy W (train_dense.hip): dy [M, K], w_t [D, K] (the layer's weight transposed, in panels), x [M, D] the
// rows in front of the norm, rstd its factor, norm_w [D] its weight. dx may be dres. dy_panels: dy is in panel order.
int dgrad_norm(const char* name, const void* dy, bool dy_panels, int32_t K, const void* w_t, const void* x, const float* rstd, const void* norm_w,
               const void* dres, void* dx, int64_t M, int32_t D, const int32_t* count, hipStream_t s);

// Weight gradients of the four dense layers of a block in one launch (train_dense.hip): G[n, k] = sum over the rows of dy[m, n] *
// a[m, k], a multiplied by scale[m] first when scale is given (a norm's factor: the norm's weight multiplies G's columns and is
// applied by the reduction). The column sums of dy ride along.
struct WgradItem {
  const bf16_t* dy;
  const bf16_t* a;
  const float* scale;       // [M] or null
  int32_t N, K;             // dy [M, N], a [M, K]
  bool dy_panels, a_panels; // ... in panel order
  // reduction: dw [N, K] = G * norm_w (per column) when norm_w is given; dnorm[k] = sum over n of w[n, k] * G[n, k]
  const void* w;            // [N, K] the layer's weight (with norm_w)
  const void* norm_w;       // [K] or null
  void* dw;
  void* db;                 // [N] or null
  void* dnorm;              // [K] or null
};
constexpr int kWgradItems = 4;
// Floats of scratch of one wgrad_block call, and of the small vectors it leaves for wgrad_vectors.
int64_t wgrad_scratch_floats(int64_t M, const int32_t (*shapes)[2], int items);
int64_t wgrad_vector_floats(int64_t M, const int32_t (*shapes)[2], int items);

// Sums of partial rows, in order: dst[c] = sum over i < parts of src[i * stride + c].
struct VectorItem {
  const float* src;
  void* dst;
  int32_t parts, stride, cols;
};
// items4[i].dw etc. are of `dtype` (TAAC_BF16 / TAAC_F32), as are w and norm_w. Appends the vectors still to be summed.
int wgrad_block(const char* name, const WgradItem* items, int n_items, int64_t M, const int32_t* count, float* scratch,
                float* vectors, int dtype, VectorItem* out_vectors, int* n_vectors, hipStream_t s);
int sum_vectors(const char* name, const VectorItem* items, int n, int dtype, hipStream_t s);

}  // namespace taac
