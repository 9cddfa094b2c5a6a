// Training stack: forward and backward of n interaction blocks (pre-RMSNorm attention with optional query / key norms, SwiGLU
// feed-forward; experiments/symbiosis/backbone.py:51-68) and, optionally, the pCVR readout behind them, each as one call that
// sequences the library's kernels on one stream.
//
// The token stream is COMPACT from the first block to the last: the valid tokens of the batch, one behind the other, gathered once
// on the way in and scattered once on the way out. The residual updates skip padded tokens (the reference multiplies them by
// ~padding_mask), so nothing in between ever looks at one: no row index in the dense kernels, no gather, merge or copy of the
// stream at block boundaries, and the attention kernels address a sample by its row offset. How many tokens there are is only
// known on the device; every kernel reads the count, grids and buffers are sized by B * T, the host never waits.
//
// The forward keeps per block: the input stream x, q | k | v, the attention output and its log-sum-exp, the stream x1 between the
// two halves, and the factors of the two norms. The backward of a block is eight launches, nine with query / key norms:
//   feed-forward backward (hidden state, gradient of the up projection)  -> x1, dy
//   input gradient of the up projection + norm backward + residual       -> dx1
//   out projection's input gradient                                       -> datt
//   attention backward (two launches; + the query / key norms')           -> dq | dk | dv
//   input gradient of the q | k | v projection + norm backward + residual -> dx
//   the four weight gradients, and the reduction of their splits (two launches)
// The normalised rows never exist in memory: the weight gradients multiply x by the norm's factor as they stage it and apply the
// norm's weight to the columns of the result; the gradient of that weight falls out of the same sums (train_ops.h).
#include <vector>

#include "pack.h"
#include "row_index.h"
#include "train_ops.h"

namespace taac {
namespace {

constexpr int kThreads = 256;
constexpr int kSetupBlocks = 16;  // blocks per set-up launch (kernel arguments)
inline int64_t align256(int64_t v) { return (v + 255) & ~static_cast<int64_t>(255); }

// ---- weights of a block, as the kernels read them -----------------------------------------------------------------------
struct PackedBlock {
  int64_t qkv, out, ffn;          // forward blobs (norm weights folded)
  int64_t ffn_bwd;                // feed-forward backward blob
  int64_t up_t, qkv_t, out_t;     // transposes [D, 2F] and [D, 3D] in dgrad_norm's order, blob of the out projection's transpose
  int64_t vectors;                // bf16: attn_norm D | qkv_bias 3D | out_bias D | ffn_norm D | up_bias 2F | down_bias D | query D | key D
  int64_t bytes;
};
PackedBlock packed_block(int32_t D, int32_t F) {
  PackedBlock b{};
  const int64_t d2 = static_cast<int64_t>(D) * D * 2, df = static_cast<int64_t>(D) * F * 2;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += align256(bytes);
    return here;
  };
  b.qkv = take(3 * d2);
  b.out = take(d2);
  b.ffn = take(3 * df);
  b.ffn_bwd = take(3 * df);
  b.up_t = take(2 * df);
  b.qkv_t = take(3 * d2);
  b.out_t = take(d2);
  b.vectors = take((static_cast<int64_t>(9) * D + 2 * F) * 2);
  b.bytes = at;
  return b;
}
struct BlockVectors {
  const bf16_t *attn_norm, *qkv_bias, *out_bias, *ffn_norm, *up_bias, *down_bias, *query_norm, *key_norm;
};
BlockVectors block_vectors(const char* packed, const PackedBlock& pb, int32_t D, int32_t F) {
  const bf16_t* v = reinterpret_cast<const bf16_t*>(packed + pb.vectors);
  return BlockVectors{v, v + D, v + 4 * D, v + 5 * D, v + 6 * D, v + 6 * D + 2 * F, v + 7 * D + 2 * F, v + 8 * D + 2 * F};
}

struct TrainSetup {
  const void* attn_norm[kSetupBlocks];
  const void* qkv[kSetupBlocks];
  const void* qkv_bias[kSetupBlocks];
  const void* out[kSetupBlocks];
  const void* out_bias[kSetupBlocks];
  const void* ffn_norm[kSetupBlocks];
  const void* up[kSetupBlocks];
  const void* up_bias[kSetupBlocks];
  const void* down[kSetupBlocks];
  const void* down_bias[kSetupBlocks];
  const void* query_norm[kSetupBlocks];
  const void* key_norm[kSetupBlocks];
  char* packed;                 // of block 0; blocks lie pb.bytes apart
  PackedBlock pb;
  int32_t D, F, gate_first;
  bool fold_act;
  uint32_t units_per_block, pack_units, row_units;
  const int32_t* lengths;       // row index, when asked for (row_units > 0)
  int32_t B, T;
  int32_t* rows;
  int32_t* n_rows;
  int32_t* clear;               // n_clear words set to zero
  int32_t n_clear;
  const void* head_w;           // [D] -> bf16 copy, or null
  bf16_t* head_w_bf16;
};

template <typename TW>
__device__ __forceinline__ void vector_piece(const TrainSetup& p, int blk, bf16_t* dst, int i) {  // entry i of the vectors
  const int D = p.D, F = p.F;
  const TW* src = nullptr;
  int at = i;
  auto segment = [&](const void* v, int n) {
    if (src == nullptr && at >= 0 && at < n) {
      src = static_cast<const TW*>(v);
      if (src == nullptr) {
        dst[i] = static_cast<bf16_t>(0.f);
        at = -1;
        return;
      }
      dst[i] = static_cast<bf16_t>(static_cast<float>(src[at]));
      at = -1;
      return;
    }
    if (at >= 0) at -= n;
  };
  segment(p.attn_norm[blk], D);
  segment(p.qkv_bias[blk], 3 * D);
  segment(p.out_bias[blk], D);
  segment(p.ffn_norm[blk], D);
  segment(p.up_bias[blk], 2 * F);
  segment(p.down_bias[blk], D);
  segment(p.query_norm[blk], D);
  segment(p.key_norm[blk], D);
}

// Piece of the transpose [cols, rows] of a row-major weight [rows, cols], in the order of dgrad_norm's weight: column d, rows c .. c + 7.
// Consecutive pieces take consecutive columns, so that the eight strided reads of a wavefront are eight contiguous runs.
template <typename TW>
__device__ __forceinline__ bf16x8 transposed_piece(const TW* w, int rows, int cols, int64_t piece, int64_t* dst) {
  const int d = static_cast<int>(piece % cols);
  const int c = static_cast<int>(piece / cols) * 8;
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(w[static_cast<int64_t>(c + e) * cols + d]));
  *dst = transposed_weight_at(d, c, cols);
  return v;
}

// Everything the forward and the backward need of the weights, and the row index, in one launch (one role per workgroup).
template <typename TW>
__global__ __launch_bounds__(kRowThreads) void train_setup_kernel(const TrainSetup p) {
  uint32_t unit = blockIdx.x;
  const int D = p.D, F = p.F;
  if (unit == 0) {
    for (int i = threadIdx.x; i < p.n_clear; i += kRowThreads) p.clear[i] = 0;
    if (p.head_w != nullptr)
      for (int i = threadIdx.x; i < D; i += kRowThreads)
        p.head_w_bf16[i] = static_cast<bf16_t>(static_cast<float>(static_cast<const TW*>(p.head_w)[i]));
  }
  if (unit >= p.pack_units) {
    unit -= p.pack_units;
    if (unit < p.row_units) write_valid_rows(p.lengths, p.B, p.T, static_cast<int>(unit), p.rows, p.n_rows);
    return;
  }
  const int blk = static_cast<int>(unit / p.units_per_block);
  char* packed = p.packed + blk * p.pb.bytes;
  const TW* qkv = static_cast<const TW*>(p.qkv[blk]);
  const TW* out = static_cast<const TW*>(p.out[blk]);
  const TW* up = static_cast<const TW*>(p.up[blk]);
  const TW* down = static_cast<const TW*>(p.down[blk]);
  const TW* attn_norm = static_cast<const TW*>(p.attn_norm[blk]);
  const TW* ffn_norm = static_cast<const TW*>(p.ffn_norm[blk]);
  const int64_t d2 = static_cast<int64_t>(D) * D / 8, df = static_cast<int64_t>(D) * F / 8;
  int64_t gid = static_cast<int64_t>(unit % p.units_per_block) * kRowThreads + threadIdx.x;
  auto blob = [&](int64_t offset) { return reinterpret_cast<bf16x8*>(packed + offset); };
  if (gid < 3 * d2) return linear_pack_piece(qkv, blob(p.pb.qkv), D, gid, attn_norm);
  gid -= 3 * d2;
  if (gid < d2) return linear_pack_piece(out, blob(p.pb.out), D, gid);
  gid -= d2;
  if (gid < 3 * df) return ffn_pack_piece(up, down, blob(p.pb.ffn), D, F, p.gate_first, gid, ffn_norm, p.fold_act);
  gid -= 3 * df;
  if (gid < 3 * df) return ffn_bwd_pack_piece(up, down, blob(p.pb.ffn_bwd), D, F, gid);
  gid -= 3 * df;
  int64_t at;
  if (gid < 2 * df) {
    const bf16x8 v = transposed_piece(up, 2 * F, D, gid, &at);
    *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16_t*>(packed + p.pb.up_t) + at) = v;
    return;
  }
  gid -= 2 * df;
  if (gid < 3 * d2) {
    const bf16x8 v = transposed_piece(qkv, 3 * D, D, gid, &at);
    *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16_t*>(packed + p.pb.qkv_t) + at) = v;
    return;
  }
  gid -= 3 * d2;
  if (gid < d2) {  // fragment order of linear_pack_piece, of the transpose: row n of it is column n of the weight
    const int KS = D / 16, NFRAG = 2 * KS;
    const int lane = static_cast<int>(gid % 64), f = static_cast<int>((gid / 64) % NFRAG);
    const int64_t chunk = gid / 64 / NFRAG;
    const int n = static_cast<int>(chunk) * kNC + (f / KS) * 32 + lane % 32, k = (f % KS) * 16 + lane / 32 * 8;
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(out[static_cast<int64_t>(k + e) * D + n]));
    blob(p.pb.out_t)[gid] = v;
    return;
  }
  gid -= d2;
  if (gid < 9 * D + 2 * F) vector_piece<TW>(p, blk, reinterpret_cast<bf16_t*>(packed + p.pb.vectors), static_cast<int>(gid));
}

// ---- rows in and out of the compact layout ------------------------------------------------------------------------------------
// dst[i] = src[rows[i]] (add: dst[i] += ...), i < *count; rows of D bf16.
__global__ __launch_bounds__(kThreads) void gather_kernel(const bf16x8* __restrict__ src, const int32_t* __restrict__ rows,
                                                          const int32_t* __restrict__ count, bf16x8* __restrict__ dst, int pieces,
                                                          int64_t M, bool add) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t i = idx / pieces;
  const int64_t n = *count;
  if (i >= (n < M ? n : M)) return;
  bf16x8 v = __builtin_nontemporal_load(src + static_cast<int64_t>(rows[i]) * pieces + idx % pieces);
  if (add) {
    const bf16x8 w = dst[idx];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) + static_cast<float>(w[e]));
  }
  dst[idx] = v;
}

// out[b, t] = compact row offsets[b] + (rank of t) for a valid token, else padded[b, t] (+ padded2[b, t]; zeros without padded).
// Valid: t < lengths[b], or bit t of the sample's validity words.
__global__ __launch_bounds__(kThreads) void scatter_kernel(const bf16x8* __restrict__ compact, const bf16x8* __restrict__ padded,
                                                           const bf16x8* __restrict__ padded2, const int32_t* __restrict__ lengths,
                                                           const uint32_t* __restrict__ valid_bits,
                                                           const int32_t* __restrict__ offsets, bf16x8* __restrict__ out,
                                                           int64_t total, int T, int pieces) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (idx >= total) return;
  const int64_t row = idx / pieces;
  const int b = static_cast<int>(row / T), t = static_cast<int>(row % T);
  int rank = -1;
  if (valid_bits == nullptr) {
    if (t < clamped_length(lengths, b, T)) rank = t;
  } else {
    const uint32_t* bits = valid_bits + static_cast<int64_t>(b) * ((T + 31) / 32);
    const uint32_t word = bits[t / 32];
    // The words in front of the row's are counted by the row's lanes together (`pieces` of them, a power of two within a wavefront): by each
    // alone it is a load behind the other, 128 x 403 tokens of 256 features 19.4 -> 14.8 us.
    const int lane = static_cast<int>(idx % pieces);
    int before = 0;
    for (int w = lane; w < t / 32; w += pieces) before += __popc(bits[w]);
    for (int off = 1; off < pieces; off <<= 1) before += __shfl_xor(before, off, kWave);
    if ((word >> (t % 32)) & 1u) rank = before + __popc(word & ((1u << (t % 32)) - 1u));
  }
  bf16x8 v;
  if (rank >= 0) {
    v = compact[(static_cast<int64_t>(offsets[b]) + rank) * pieces + idx % pieces];
  } else if (padded != nullptr) {
    v = padded[idx];
    if (padded2 != nullptr) {
      const bf16x8 w = padded2[idx];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) + static_cast<float>(w[e]));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(0.f);
  }
  out[idx] = v;
}

// ---- readout --------------------------------------------------------------------------------------------------------------------
// p[b] = sigmoid(mean of the sample's token dots + bias): one wavefront per sample, fixed order.
template <typename TW>
__global__ __launch_bounds__(kThreads) void compact_head_kernel(const float* __restrict__ dots, const int32_t* __restrict__ offsets,
                                                                const TW* __restrict__ b_head, float* __restrict__ p, int B) {
  const int b = blockIdx.x * (kThreads / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  if (b >= B) return;
  const int begin = offsets[b], len = offsets[b + 1] - begin;
  float s = 0.f;
  for (int t = lane; t < len; t += kWave) s += dots[begin + t];
  s = group_sum<kWave>(s);
  if (lane == 0) {
    const float z = (b_head != nullptr ? static_cast<float>(static_cast<bf16_t>(static_cast<float>(b_head[0]))) : 0.f) +
                    s / static_cast<float>(len < 1 ? 1 : len);
    p[b] = 1.0f / (1.0f + expf(-z));
  }
}

// Backward of the readout, one workgroup per sample: c = dp p (1 - p) / len; every row of the sample receives c * w_head, the
// sample's share of the weight gradient is c * (sum of its rows), of the bias gradient dp p (1 - p).
__global__ __launch_bounds__(kThreads) void head_bwd_kernel(const bf16_t* __restrict__ x, const float* __restrict__ dp,
                                                            const float* __restrict__ p, const int32_t* __restrict__ offsets,
                                                            const bf16_t* __restrict__ w_head, bf16_t* __restrict__ dy,
                                                            float* __restrict__ dw_part, float* __restrict__ db_part, int D) {
  __shared__ float acc_lds[kThreads][8];
  const int b = blockIdx.x;
  const int begin = offsets[b], len = offsets[b + 1] - begin;
  const int c8n = D / 8, groups = kThreads / c8n;
  const int chunk = threadIdx.x % c8n, group = threadIdx.x / c8n;
  const float dz = dp[b] * p[b] * (1.f - p[b]);
  const float c = dz / static_cast<float>(len < 1 ? 1 : len);
  const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w_head + chunk * 8);
  bf16x8 grad;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    grad[e] = static_cast<bf16_t>(c * static_cast<float>(wv[e]));
    acc[e] = 0.f;
  }
#pragma unroll 4
  for (int t = group; t < len; t += groups) {
    const int64_t at = (static_cast<int64_t>(begin) + t) * D + chunk * 8;
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(x + at);
    *reinterpret_cast<bf16x8*>(dy + at) = grad;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += static_cast<float>(v[e]);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) acc_lds[threadIdx.x][e] = acc[e];
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += kThreads) {
    float s = 0.f;
    for (int g = 0; g < groups; ++g) s += acc_lds[g * c8n + d / 8][d % 8];
    dw_part[static_cast<int64_t>(b) * D + d] = c * s;
  }
  if (threadIdx.x == 0) db_part[b] = dz;
}

// ---- query / key norms ------------------------------------------------------------------------------------------------------------
// out [M, 2D] = rmsnorm(q) | rmsnorm(k) of the packed rows qkv [M, 3D], each over its D features. D / 8 lanes per (token, part).
template <int D>
__global__ __launch_bounds__(kThreads) void qk_norm_kernel(const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ wq,
                                                           const bf16_t* __restrict__ wk, float eps, bf16_t* __restrict__ out,
                                                           const int32_t* __restrict__ count, int64_t M) {
  constexpr int G = D / 8;
  const int lane = threadIdx.x % G;
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * (kThreads / G) + threadIdx.x / G;
  const int64_t n = *count;
  const int64_t m = unit >> 1;
  const int part = static_cast<int>(unit & 1);
  if (m >= (n < M ? n : M)) return;
  const bf16x8 v = *reinterpret_cast<const bf16x8*>(qkv + m * (3 * D) + part * D + lane * 8);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(static_cast<float>(v[e]), static_cast<float>(v[e]), ss);
  const float r = rsqrtf(group_sum<G>(ss) * (1.0f / D) + eps);
  const bf16x8 w = *reinterpret_cast<const bf16x8*>((part == 0 ? wq : wk) + lane * 8);
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = static_cast<bf16_t>(static_cast<float>(v[e]) * r * static_cast<float>(w[e]));
  *reinterpret_cast<bf16x8*>(out + m * (2 * D) + part * D + lane * 8) = o;
}

// Their backward, in place on the q | k columns of dqkv [M, 3D]; per workgroup the sums of g * x_hat in dw_part [gridDim.x][2D].
constexpr int kQkBlocks = 512;
template <int D>
__global__ __launch_bounds__(kThreads) void qk_norm_bwd_kernel(const bf16_t* __restrict__ qkv, bf16_t* __restrict__ dqkv,
                                                               const bf16_t* __restrict__ wq, const bf16_t* __restrict__ wk,
                                                               float eps, float* __restrict__ dw_part,
                                                               const int32_t* __restrict__ count, int64_t M) {
  constexpr int G = D / 8, GPB = kThreads / G;  // lane groups per workgroup: even ones take queries, odd ones keys
  __shared__ float red[GPB][D];
  const int lane = threadIdx.x % G, gid = threadIdx.x / G;
  const int part = gid & 1;
  int64_t rows = *count;
  rows = rows < M ? rows : M;
  const bf16x8 wv = *reinterpret_cast<const bf16x8*>((part == 0 ? wq : wk) + lane * 8);
  float w[8], dw[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    w[e] = static_cast<float>(wv[e]);
    dw[e] = 0.f;
  }
  constexpr int R = 2;
  constexpr int64_t kStep = GPB / 2;
  // The rows of the next step are requested in front of this step's: behind its stores they would wait for those as well (loads and
  // stores complete in one order), a memory latency and the stores in every step (29 000
  // rows of 256, us: 23.2 -> 17.8).
  const int64_t stride = static_cast<int64_t>(gridDim.x) * R * kStep;
  const int64_t first = (static_cast<int64_t>(blockIdx.x) * R) * kStep + gid / 2;
  auto request = [&](int64_t m0, bf16x8 (&xv)[R], bf16x8 (&gv)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t m = m0 + r * kStep;
      const int64_t at = (m < rows ? m : first) * (3 * D) + part * D + lane * 8;  // (its values are not used then)
      xv[r] = *reinterpret_cast<const bf16x8*>(qkv + at);
      gv[r] = *reinterpret_cast<const bf16x8*>(dqkv + at);
    }
  };
  auto step = [&](int64_t m0, const bf16x8 (&xv)[R], const bf16x8 (&gv)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (m0 + r * kStep >= rows) continue;  // the same for the whole lane group
      float ss = 0.f, sg = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = static_cast<float>(xv[r][e]);
        ss = fmaf(x, x, ss);
        sg = fmaf(static_cast<float>(gv[r][e]) * w[e], x, sg);
      }
      const float rstd = rsqrtf(group_sum<G>(ss) * (1.0f / D) + eps);
      const float proj = group_sum<G>(sg) * (1.0f / D) * rstd * rstd;
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = static_cast<float>(xv[r][e]), g = static_cast<float>(gv[r][e]);
        o[e] = static_cast<bf16_t>(rstd * (g * w[e] - x * proj));
        dw[e] = fmaf(g, x * rstd, dw[e]);
      }
      *reinterpret_cast<bf16x8*>(dqkv + (m0 + r * kStep) * (3 * D) + part * D + lane * 8) = o;
    }
  };
  if (first < rows) {
    bf16x8 xa[R], ga[R], xb[R], gb[R];
    request(first, xa, ga);
    for (int64_t m0 = first; m0 < rows; m0 += 2 * stride) {
      request(m0 + stride, xb, gb);
      __builtin_amdgcn_sched_barrier(0);
      step(m0, xa, ga);
      request(m0 + 2 * stride, xa, ga);
      __builtin_amdgcn_sched_barrier(0);
      step(m0 + stride, xb, gb);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[gid][lane * 8 + e] = dw[e];
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * D; i += kThreads) {
    float s = 0.f;
#pragma unroll
    for (int g = i / D; g < GPB; g += 2) s += red[g][i % D];
    dw_part[static_cast<int64_t>(blockIdx.x) * (2 * D) + i] = s;
  }
}

// ---- buffers ------------------------------------------------------------------------------------------------------------------
struct Sizes {
  int32_t B, T, D, H, F, n;
  bool qk;
  int64_t M;
  int32_t shapes[kWgradItems][2];
};
Sizes sizes_of(int32_t B, int32_t T, int32_t D, int32_t H, int32_t F, int32_t n, int qk) {
  Sizes z{B, T, D, H, F, n, qk != 0, static_cast<int64_t>(B) * T, {{3 * D, D}, {D, D}, {2 * F, D}, {D, F}}};
  return z;
}

// What a forward leaves for its backward.
struct Saved {
  int32_t* rows;      // [M] + offsets [B + 1]
  int32_t* count;
  char* packed;
  PackedBlock pb;
  bf16_t* head_w;     // bf16 copy
  struct Block {
    bf16_t *x, *qkv, *att, *x1, *qk;
    float *lse, *rstd_attn, *rstd_ffn;
  };
  std::vector<Block> block;
  bf16_t* x_last;
  int64_t bytes;
};
Saved saved_layout(const Sizes& z, char* base) {
  Saved s{};
  char* at = base;
  auto take = [&](int64_t bytes) {
    char* here = at;
    at += align256(bytes);
    return here;
  };
  s.rows = reinterpret_cast<int32_t*>(take((z.M + z.B + 2) * 4));
  s.count = s.rows + z.M + z.B + 1;
  s.pb = packed_block(z.D, z.F);
  s.packed = take(s.pb.bytes * z.n);
  s.head_w = reinterpret_cast<bf16_t*>(take(z.D * 2));
  const int64_t row = z.M * z.D * 2;
  for (int i = 0; i < z.n; ++i) {
    Saved::Block b{};
    b.x = reinterpret_cast<bf16_t*>(take(row));
    b.qkv = reinterpret_cast<bf16_t*>(take(3 * row));
    b.att = reinterpret_cast<bf16_t*>(take(row));
    b.x1 = reinterpret_cast<bf16_t*>(take(row));
    b.qk = z.qk ? reinterpret_cast<bf16_t*>(take(2 * row)) : nullptr;
    b.lse = reinterpret_cast<float*>(take(static_cast<int64_t>(z.B) * z.H * z.T * 4));
    b.rstd_attn = reinterpret_cast<float*>(take(z.M * 4));
    b.rstd_ffn = reinterpret_cast<float*>(take(z.M * 4));
    s.block.push_back(b);
  }
  s.x_last = reinterpret_cast<bf16_t*>(take(row));
  s.bytes = at - base;
  return s;
}

struct Scratch {
  // forward
  float* token_dots;
  char* split;
  // backward
  bf16_t *dy, *dx1, *hidden, *grad_pre, *datt, *dqkv;
  float *delta, *wgrad, *vectors, *qk_part, *head_part;
  int64_t vector_stride, bytes;
};
Scratch scratch_layout(const Sizes& z, char* base, bool backward) {
  Scratch s{};
  char* at = base;
  auto take = [&](int64_t bytes) {
    char* here = at;
    at += align256(bytes);
    return here;
  };
  if (!backward) {
    s.token_dots = reinterpret_cast<float*>(take(z.M * 4));
    s.split = take(ffn_split_bytes(z.M, z.D, z.F));
  } else {
    const int64_t row = z.M * z.D * 2;
    s.dy = reinterpret_cast<bf16_t*>(take(row));
    s.dx1 = reinterpret_cast<bf16_t*>(take(row));
    s.hidden = reinterpret_cast<bf16_t*>(take(panel_rows(z.M) * z.F * 2));  // panel order
    s.grad_pre = reinterpret_cast<bf16_t*>(take(panel_rows(z.M) * z.F * 4));
    s.datt = reinterpret_cast<bf16_t*>(take(row));
    s.dqkv = reinterpret_cast<bf16_t*>(take(3 * row));
    s.delta = reinterpret_cast<float*>(take(static_cast<int64_t>(z.B) * z.H * z.T * 4));
    // (two items where no gradient reaches the feed-forward half: more splits of fewer tiles)
    const int64_t w4 = wgrad_scratch_floats(z.M, z.shapes, kWgradItems), w2 = wgrad_scratch_floats(z.M, z.shapes, 2);
    const int64_t v4 = wgrad_vector_floats(z.M, z.shapes, kWgradItems), v2 = wgrad_vector_floats(z.M, z.shapes, 2);
    s.wgrad = reinterpret_cast<float*>(take((w4 > w2 ? w4 : w2) * 4));
    s.vector_stride = v4 > v2 ? v4 : v2;
    s.vectors = reinterpret_cast<float*>(take(s.vector_stride * z.n * 4));
    s.qk_part = reinterpret_cast<float*>(take(z.qk ? static_cast<int64_t>(z.n) * kQkBlocks * 2 * z.D * 4 : 0));
    s.head_part = reinterpret_cast<float*>(take((static_cast<int64_t>(z.B) * (z.D + 1)) * 4));
  }
  s.bytes = at - base;
  return s;
}

bool shape_ok(const Sizes& z) {
  return (z.D == 128 || z.D == 256) && z.H > 0 && z.D % z.H == 0 && (z.D / z.H == 32 || z.D / z.H == 64) && z.F > 0 && z.F % 32 == 0 &&
         taac_swiglu_ffn_bwd_packed_bytes(z.D, z.F) >= 0 && z.n > 0 && z.B > 0 && z.T > 0 && z.M <= 0x7fffffffLL - z.B - 2;
}

uint32_t grid_of(int64_t threads) { return static_cast<uint32_t>((threads + kThreads - 1) / kThreads); }

}  // namespace
}  // namespace taac

extern "C" int64_t taac_stack_train_bytes(int32_t B, int32_t T, int32_t D, int32_t H, int32_t F, int32_t n_blocks, int qk_norm,
                                          int what) {
  using namespace taac;
  if (B < 0 || T < 0 || D <= 0 || H <= 0 || F <= 0 || n_blocks <= 0) return -1;
  const Sizes z = sizes_of(B, T, D, H, F, n_blocks, qk_norm);
  if (!shape_ok(z)) return -1;
  if (what == 0) return saved_layout(z, nullptr).bytes;
  return scratch_layout(z, nullptr, what == 2).bytes + 256;
}

extern "C" int taac_stack_train_fwd(const void* tokens, const int32_t* key_lengths, const int32_t* rows_given,
                                    const int32_t* count_given, const uint32_t* valid_bits, const uint32_t* struct_bits,
                                    int64_t struct_sample_stride, const taac_block_weights* blocks, int32_t n_blocks,
                                    int param_dtype, int32_t B, int32_t T, int32_t D, int32_t H, int32_t F, float attn_eps,
                                    float ffn_eps, float qk_eps, int gate_first, const void* head_w, const void* head_b,
                                    void* saved, void* scratch, void* out, int zero_padded_rows, void* attn_tokens_out, float* p,
                                    void* stream) {
  using namespace taac;
  const char* name = "taac_stack_train_fwd";
  if (B < 0 || T < 0 || D <= 0 || H <= 0 || F <= 0 || n_blocks <= 0 || !blocks)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  const Sizes z = sizes_of(B, T, D, H, F, n_blocks, blocks[0].query_norm_weight != nullptr);
  if (!shape_ok(z)) return set_error(TAAC_ERR_UNSUPPORTED, "%s: shape not covered (see taac_stack_train_bytes)", name);
  if (param_dtype != TAAC_BF16 && param_dtype != TAAC_F32)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: parameters are bf16 or fp32", name);
  if (!tokens || !key_lengths || !saved || !scratch || (struct_bits && (!rows_given || !count_given || !valid_bits)) ||
      ((p == nullptr) != (head_w == nullptr)))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(tokens) || !aligned16(out) || !aligned16(attn_tokens_out) || (reinterpret_cast<uintptr_t>(saved) & 255u) ||
      (reinterpret_cast<uintptr_t>(scratch) & 255u))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: tensors must be 16-byte, the buffers 256-byte aligned", name);
  hipStream_t s = as_stream(stream);
  Saved sv = saved_layout(z, static_cast<char*>(saved));
  Scratch sc = scratch_layout(z, static_cast<char*>(scratch), false);
  const int64_t M = z.M;
  const bool fold_act = gate_first && ffn_act_fold_supported(D, F);

  const int32_t* rows = rows_given != nullptr ? rows_given : sv.rows;
  const int32_t* count = rows_given != nullptr ? count_given : sv.count;
  const int32_t* offsets = rows + M;
  int rc = TAAC_OK;
  const bool index_in_setup = rows_given == nullptr && row_index_in_one_launch(B, T, false);
  if (rows_given == nullptr && !index_in_setup && (rc = taac_valid_rows(key_lengths, B, T, sv.rows, sv.count, stream)) != TAAC_OK)
    return rc;
  for (int first = 0; first < n_blocks; first += kSetupBlocks) {
    TrainSetup t{};
    const int n = n_blocks - first < kSetupBlocks ? n_blocks - first : kSetupBlocks;
    for (int i = 0; i < n; ++i) {
      const taac_block_weights& w = blocks[first + i];
      if (!w.attn_norm_weight || !w.qkv_weight || !w.out_weight || !w.ffn_norm_weight || !w.up_weight || !w.down_weight ||
          (w.query_norm_weight != nullptr) != z.qk || (w.key_norm_weight != nullptr) != z.qk)
        return set_error(TAAC_ERR_INVALID_VALUE, "%s: block %d has a null weight", name, first + i);
      const void* ptrs[6] = {w.attn_norm_weight, w.qkv_weight, w.out_weight, w.ffn_norm_weight, w.up_weight, w.down_weight};
      for (const void* ptr : ptrs)
        if (!aligned16(ptr)) return set_error(TAAC_ERR_UNSUPPORTED, "%s: weights must be 16-byte aligned", name);
      t.attn_norm[i] = w.attn_norm_weight;
      t.qkv[i] = w.qkv_weight;
      t.qkv_bias[i] = w.qkv_bias;
      t.out[i] = w.out_weight;
      t.out_bias[i] = w.out_bias;
      t.ffn_norm[i] = w.ffn_norm_weight;
      t.up[i] = w.up_weight;
      t.up_bias[i] = w.up_bias;
      t.down[i] = w.down_weight;
      t.down_bias[i] = w.down_bias;
      t.query_norm[i] = w.query_norm_weight;
      t.key_norm[i] = w.key_norm_weight;
    }
    t.packed = sv.packed + first * sv.pb.bytes;
    t.pb = sv.pb;
    t.D = D;
    t.F = F;
    t.gate_first = gate_first ? 1 : 0;
    t.fold_act = fold_act;
    const int64_t pieces = (8LL * D * D + 8LL * D * F) / 8 + 9 * D + 2 * F;
    t.units_per_block = static_cast<uint32_t>((pieces + kRowThreads - 1) / kRowThreads);
    t.pack_units = t.units_per_block * n;
    t.lengths = key_lengths;
    t.B = B;
    t.T = T;
    if (first == 0) {
      if (index_in_setup) {
        t.rows = sv.rows;
        t.n_rows = sv.count;
        t.row_units = static_cast<uint32_t>(B) * (T > kRowThreads ? (T + kRowThreads - 1) / kRowThreads : 1);
      }
      if (const int splits = ffn_splits(M, D, F); splits > 1) {
        const int64_t tiles = (M + 31) / 32;
        t.clear = reinterpret_cast<int32_t*>(sc.split + tiles * splits * 32 * D * 4);
        t.n_clear = static_cast<int32_t>(tiles);
      }
      t.head_w = head_w;
      t.head_w_bf16 = sv.head_w;
    }
    const dim3 setup_grid(t.pack_units + t.row_units);
    if (param_dtype == TAAC_F32)
      hipLaunchKernelGGL(train_setup_kernel<float>, setup_grid, dim3(kRowThreads), 0, s, t);
    else
      hipLaunchKernelGGL(train_setup_kernel<bf16_t>, setup_grid, dim3(kRowThreads), 0, s, t);
    if ((rc = check_launch(name)) != TAAC_OK) return rc;
  }
  const int c8 = D / 8;
  hipLaunchKernelGGL(gather_kernel, dim3(grid_of(M * c8)), dim3(kThreads), 0, s, static_cast<const bf16x8*>(tokens), rows, count,
                     reinterpret_cast<bf16x8*>(sv.block[0].x), c8, M, false);
  if ((rc = check_launch(name)) != TAAC_OK) return rc;
  char* split = ffn_split_bytes(M, D, F) > 0 ? sc.split : nullptr;
  for (int i = 0; i < n_blocks; ++i) {
    const Saved::Block& b = sv.block[i];
    const char* pk = sv.packed + i * sv.pb.bytes;
    const BlockVectors v = block_vectors(pk, sv.pb, D, F);
    bf16_t* next = i + 1 < n_blocks ? sv.block[i + 1].x : sv.x_last;
    if ((rc = norm_linear_count(name, b.x, v.attn_norm, attn_eps, v.qkv_bias, pk + sv.pb.qkv, b.qkv, M, 3 * D, D, count, b.rstd_attn,
                                s)) != TAAC_OK)
      return rc;
    if (z.qk) {
      const dim3 grid(grid_of(2 * M * c8));
      if (D == 256)
        hipLaunchKernelGGL(qk_norm_kernel<256>, grid, dim3(kThreads), 0, s, b.qkv, v.query_norm, v.key_norm, qk_eps, b.qk, count, M);
      else
        hipLaunchKernelGGL(qk_norm_kernel<128>, grid, dim3(kThreads), 0, s, b.qkv, v.query_norm, v.key_norm, qk_eps, b.qk, count, M);
      if ((rc = check_launch(name)) != TAAC_OK) return rc;
    }
    if ((rc = attention_compact_fwd(name, z.qk ? b.qk : b.qkv, b.qkv + 2 * D, z.qk ? 2 * D : 3 * D, 3 * D, key_lengths, offsets,
                                    struct_bits, struct_sample_stride, b.att, D, b.lse, B, H, T, D / H, s)) != TAAC_OK)
      return rc;
    const bool ride = i == n_blocks - 1 && p != nullptr;
    if ((rc = attn_out_ffn_count(name, b.att, v.out_bias, pk + sv.pb.out, b.x, v.ffn_norm, ffn_eps, v.up_bias, v.down_bias,
                                 pk + sv.pb.ffn, next, b.x1, b.rstd_ffn, M, D, F, gate_first != 0, fold_act, count,
                                 ride ? sv.head_w : nullptr, ride ? sc.token_dots : nullptr, split, s)) != TAAC_OK)
      return rc;
  }
  if (p != nullptr) {
    const dim3 grid((B + kThreads / kWave - 1) / (kThreads / kWave));
    if (param_dtype == TAAC_F32)
      hipLaunchKernelGGL(compact_head_kernel<float>, grid, dim3(kThreads), 0, s, sc.token_dots, offsets,
                         static_cast<const float*>(head_b), p, B);
    else
      hipLaunchKernelGGL(compact_head_kernel<bf16_t>, grid, dim3(kThreads), 0, s, sc.token_dots, offsets,
                         static_cast<const bf16_t*>(head_b), p, B);
    if ((rc = check_launch(name)) != TAAC_OK) return rc;
  }
  const int64_t total = M * c8;
  auto scatter = [&](const bf16_t* compact, void* dst) {
    hipLaunchKernelGGL(scatter_kernel, dim3(grid_of(total)), dim3(kThreads), 0, s, reinterpret_cast<const bf16x8*>(compact),
                       zero_padded_rows ? nullptr : static_cast<const bf16x8*>(tokens), static_cast<const bf16x8*>(nullptr),
                       key_lengths, valid_bits, offsets, static_cast<bf16x8*>(dst), total, T, c8);
    return check_launch(name);
  };
  if (out != nullptr && (rc = scatter(sv.x_last, out)) != TAAC_OK) return rc;
  if (attn_tokens_out != nullptr && (rc = scatter(sv.block[n_blocks - 1].x1, attn_tokens_out)) != TAAC_OK) return rc;
  return TAAC_OK;
}

extern "C" int taac_stack_train_bwd(const void* grad_out, const void* grad_attn_tokens, const float* grad_p, const float* p,
                                    const int32_t* key_lengths, const int32_t* rows_given, const int32_t* count_given,
                                    const uint32_t* valid_bits, const uint32_t* struct_bits, int64_t struct_sample_stride,
                                    const taac_block_weights* blocks, const taac_block_weights* grads, int32_t n_blocks,
                                    int param_dtype, int32_t B, int32_t T, int32_t D, int32_t H, int32_t F, float qk_eps,
                                    int gate_first, void* grad_head_w, void* grad_head_b, int zero_padded_rows, const void* saved,
                                    void* scratch, void* grad_tokens, void* stream) {
  using namespace taac;
  const char* name = "taac_stack_train_bwd";
  if (B < 0 || T < 0 || D <= 0 || H <= 0 || F <= 0 || n_blocks <= 0 || !blocks || !grads)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  const Sizes z = sizes_of(B, T, D, H, F, n_blocks, blocks[0].query_norm_weight != nullptr);
  if (!shape_ok(z)) return set_error(TAAC_ERR_UNSUPPORTED, "%s: shape not covered (see taac_stack_train_bytes)", name);
  if (param_dtype != TAAC_BF16 && param_dtype != TAAC_F32)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: parameters are bf16 or fp32", name);
  if (!key_lengths || !saved || !scratch || (grad_p != nullptr && (!p || !grad_head_w)) ||
      (grad_p == nullptr && grad_out == nullptr && grad_attn_tokens == nullptr) ||
      (struct_bits && (!rows_given || !count_given || !valid_bits)))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(grad_out) || !aligned16(grad_attn_tokens) || !aligned16(grad_tokens) || (reinterpret_cast<uintptr_t>(saved) & 255u) ||
      (reinterpret_cast<uintptr_t>(scratch) & 255u))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: tensors must be 16-byte, the buffers 256-byte aligned", name);
  hipStream_t s = as_stream(stream);
  const Saved sv = saved_layout(z, static_cast<char*>(const_cast<void*>(saved)));
  const Scratch sc = scratch_layout(z, static_cast<char*>(scratch), true);
  const int64_t M = z.M;
  const int32_t* rows = rows_given != nullptr ? rows_given : sv.rows;
  const int32_t* count = rows_given != nullptr ? count_given : sv.count;
  const int32_t* offsets = rows + M;
  const int c8 = D / 8;
  int rc = TAAC_OK;
  std::vector<VectorItem> vectors(static_cast<size_t>(n_blocks) * 10 + 2);
  int n_vectors = 0;
  auto gather = [&](const void* src, bf16_t* dst, bool add) {
    hipLaunchKernelGGL(gather_kernel, dim3(grid_of(M * c8)), dim3(kThreads), 0, s, static_cast<const bf16x8*>(src), rows, count,
                       reinterpret_cast<bf16x8*>(dst), c8, M, add);
    return check_launch(name);
  };
  bf16_t* dy = sc.dy;
  bool have_dy = false;
  if (grad_p != nullptr) {
    float* dw_part = sc.head_part;
    float* db_part = sc.head_part + static_cast<int64_t>(B) * D;
    hipLaunchKernelGGL(head_bwd_kernel, dim3(B), dim3(kThreads), 0, s, sv.x_last, grad_p, p, offsets, sv.head_w, dy, dw_part, db_part, D);
    if ((rc = check_launch(name)) != TAAC_OK) return rc;
    vectors[n_vectors++] = VectorItem{dw_part, grad_head_w, B, D, D};
    if (grad_head_b != nullptr) vectors[n_vectors++] = VectorItem{db_part, grad_head_b, B, 1, 1};
    have_dy = true;
  }
  if (grad_out != nullptr) {
    if ((rc = gather(grad_out, dy, have_dy)) != TAAC_OK) return rc;
    have_dy = true;
  }
  for (int i = n_blocks - 1; i >= 0; --i) {
    const Saved::Block& b = sv.block[i];
    const char* pk = sv.packed + i * sv.pb.bytes;
    const BlockVectors v = block_vectors(pk, sv.pb, D, F);
    const taac_block_weights& w = blocks[i];
    const taac_block_weights& g = grads[i];
    bf16_t* dx1 = sc.dx1;
    if (have_dy) {
      if ((rc = ffn_bwd_hidden_count(name, b.x1, b.rstd_ffn, v.ffn_norm, dy, pk + sv.pb.ffn_bwd, v.up_bias, sc.hidden, sc.grad_pre, M, D, F,
                                     gate_first != 0, count, s)) != TAAC_OK)
        return rc;
      if ((rc = dgrad_norm(name, sc.grad_pre, true, 2 * F, pk + sv.pb.up_t, b.x1, b.rstd_ffn, v.ffn_norm, dy, dx1, M, D, count, s)) != TAAC_OK)
        return rc;
    }
    // (a gradient of the tokens between the halves belongs to a stack of one block)
    if (grad_attn_tokens != nullptr && (rc = gather(grad_attn_tokens, dx1, have_dy)) != TAAC_OK) return rc;
    if ((rc = norm_linear_count(name, dx1, nullptr, 0.f, nullptr, pk + sv.pb.out_t, sc.datt, M, D, D, count, nullptr, s)) != TAAC_OK)
      return rc;
    if ((rc = attention_compact_bwd(name, z.qk ? b.qk : b.qkv, b.qkv + 2 * D, z.qk ? 2 * D : 3 * D, 3 * D, b.att, D, sc.datt, D, b.lse,
                                    key_lengths, offsets, struct_bits, struct_sample_stride, sc.dqkv, 3 * D, sc.delta, B, H, T,
                                    D / H, s)) != TAAC_OK)
      return rc;
    if (z.qk) {
      const int64_t per = 2 * (kThreads / c8) / 2;  // tokens per workgroup and step
      int64_t nb = (M + per - 1) / per;
      if (nb > kQkBlocks) nb = kQkBlocks;
      float* part = sc.qk_part + static_cast<int64_t>(i) * kQkBlocks * 2 * D;
      if (D == 256)
        hipLaunchKernelGGL(qk_norm_bwd_kernel<256>, dim3(static_cast<uint32_t>(nb)), dim3(kThreads), 0, s, b.qkv, sc.dqkv,
                           v.query_norm, v.key_norm, qk_eps, part, count, M);
      else
        hipLaunchKernelGGL(qk_norm_bwd_kernel<128>, dim3(static_cast<uint32_t>(nb)), dim3(kThreads), 0, s, b.qkv, sc.dqkv,
                           v.query_norm, v.key_norm, qk_eps, part, count, M);
      if ((rc = check_launch(name)) != TAAC_OK) return rc;
      vectors[n_vectors++] = VectorItem{part, const_cast<void*>(g.query_norm_weight), static_cast<int32_t>(nb), 2 * D, D};
      vectors[n_vectors++] = VectorItem{part + D, const_cast<void*>(g.key_norm_weight), static_cast<int32_t>(nb), 2 * D, D};
    }
    WgradItem items[kWgradItems] = {
        {sc.dqkv, b.x, b.rstd_attn, 3 * D, D, false, false, w.qkv_weight, w.attn_norm_weight, const_cast<void*>(g.qkv_weight),
         const_cast<void*>(g.qkv_bias), const_cast<void*>(g.attn_norm_weight)},
        {dx1, b.att, nullptr, D, D, false, false, nullptr, nullptr, const_cast<void*>(g.out_weight), const_cast<void*>(g.out_bias), nullptr},
        {sc.grad_pre, b.x1, b.rstd_ffn, 2 * F, D, true, false, w.up_weight, w.ffn_norm_weight, const_cast<void*>(g.up_weight),
         const_cast<void*>(g.up_bias), const_cast<void*>(g.ffn_norm_weight)},
        {dy, sc.hidden, nullptr, D, F, false, true, nullptr, nullptr, const_cast<void*>(g.down_weight), const_cast<void*>(g.down_bias), nullptr}};
    if ((rc = wgrad_block(name, items, have_dy ? 4 : 2, M, count, sc.wgrad, sc.vectors + i * sc.vector_stride, param_dtype,
                          vectors.data(), &n_vectors, s)) != TAAC_OK)
      return rc;
    // the block's input gradient takes the place of dy, which nothing reads any more
    if ((i > 0 || grad_tokens != nullptr) &&
        (rc = dgrad_norm(name, sc.dqkv, false, 3 * D, pk + sv.pb.qkv_t, b.x, b.rstd_attn, v.attn_norm, dx1, dy, M, D, count, s)) != TAAC_OK)
      return rc;
    have_dy = true;
  }
  if ((rc = sum_vectors(name, vectors.data(), n_vectors, param_dtype, s)) != TAAC_OK) return rc;
  if (grad_tokens == nullptr) return TAAC_OK;
  const int64_t total = M * c8;
  const void* padded = zero_padded_rows ? nullptr : (grad_out != nullptr ? grad_out : grad_attn_tokens);
  const void* padded2 = zero_padded_rows || grad_out == nullptr ? nullptr : grad_attn_tokens;
  hipLaunchKernelGGL(scatter_kernel, dim3(grid_of(total)), dim3(kThreads), 0, s, reinterpret_cast<const bf16x8*>(dy),
                     static_cast<const bf16x8*>(padded), static_cast<const bf16x8*>(padded2), key_lengths, valid_bits, offsets,
                     static_cast<bf16x8*>(grad_tokens), total, T, c8);
  return check_launch(name);
}
