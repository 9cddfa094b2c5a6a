// Parameters and device pieces shared by the token-stationary dense kernels (ffn.hip: a workgroup keeps hundreds of tokens
// and the weights stream past them; ffn_small.hip: few tokens, the weights spread over the wavefronts).
#pragma once

#include "common.h"
#include "ts_common.h"

namespace taac {
namespace {

constexpr int kFrag = 1024;  // bytes of one 32 x 16 bf16 MFMA operand fragment
constexpr int kNC = 64;      // output features per chunk of the plain linear kernel
constexpr int kHU = 16;      // hidden units per FFN chunk
constexpr int kCPB = 2;      // FFN chunks per barrier step
constexpr int kStageRow = kNC * 2 + 16;       // bytes per token row of the epilogue tile (64 features + pad)
constexpr int kStageWave = 32 * kStageRow;    // epilogue tile of one wavefront: 32 tokens x 64 features

}  // namespace

constexpr int kMaxLdsBytes = 160 * 1024;  // of a compute unit

struct TsParams {
  const bf16_t* x;          // [M, D] row stride ldx
  const bf16_t* norm_w;     // [D] or null (no normalisation)
  const bf16_t* w1;         // FFN: w_up [2F, D] or the packed blob; linear: w [N, D] or the packed blob
  const bf16_t* b1;         // FFN: b_up [2F] or null; linear: bias [N] or null
  const bf16_t* w2;         // FFN: w_down [D, F] (unused when packed)
  const bf16_t* b2;         // FFN: b_down [D] or null
  const bf16_t* residual;   // [M, D or N] row stride ldr, or null
  bf16_t* out;              // [M, D or N] row stride ldo
  int64_t M, ldx, ldr, ldo;
  int32_t F;                // FFN hidden size
  int32_t N;                // linear output features
  float eps;
  int32_t gate_first;
  int32_t packed;           // weights are in fragment order
  const int32_t* rows;      // optional row index: token i lives in row rows[i] of x / residual / out
  const int32_t* n_rows;    // device pointer to the number of tokens (at most M), or null: M. Without rows the tokens are the
                            // first *n_rows rows (a compact tensor whose length the host does not know)
  const int32_t* x_rows;    // optional, with rows: token i's row of x when it differs from rows[i] (x and residual / out
                            // laid out differently: samples with their valid tokens moved to the front on one side)
  int32_t units;            // FFN: compute units the last, partial round of workgroups is spread over; few-token kernel: its workgroups
                            // that run at once
  // Query / key mode of the linear kernel (the packed q | k | v projection of an attention layer):
  const bf16_t* qk_w;       // [D] norm weight of the query features, or null (ones)
  const bf16_t* qk_wk;      // [D] norm weight of the key features, with qk_w
  const bf16_t* cos_sin;    // rotary table [tokens_per_sample][head_dim] of (cos, sin) pairs, or null
  float* qk_sumsq;          // [qk_chunks][M] sum of squares of a token's 64 features of one chunk
  float* qk_rstd;           // [2][M] factors of the query and key norm, or null. Given, it takes the place of qk_sumsq, which the
                            // persistent kernel then uses for the token tiles whose chunks it divides over workgroups
  uint32_t* qk_counters;    // persistent kernel, with qk_rstd: [kQkCounters], zero before the launch and behind it
  float qk_eps;
  int32_t qk_chunks;        // leading 64-feature chunks that belong to the query and key projections
  int32_t head_dim, tokens_per_sample;
  // Attention output projection in front of the FFN (x is then the attention output, residual the block input):
  const bf16_t* w0;         // packed [D, D] projection (linear blob)
  const bf16_t* b0;         // its bias [D] or null
  int32_t norm_folded;      // linear kernel: norm_w is already part of the packed weights (taac_linear_pack_weights_norm):
                            // the rows enter the products as they are and only the factor rsqrt(mean + eps) is applied, to the
                            // accumulators
  const bf16_t* gate;       // GATE: [M, D] pre-activation of the update's gate (rows like residual), row stride ldg
  int64_t ldg;
  // Feature planes (the backbone's private q | k | v and attention-output buffers): with a shift s > 0 the tensor is a
  // stack of planes of 2^s features, [cols / 2^s][M][2^s] - element (row, col) at ((col >> s) * M + row) * 2^s + col % 2^s -
  // instead of [M][cols] rows; a head's rows are then contiguous for the attention kernel.
  int32_t x_plane_shift;    // layout of x (0: rows of ldx elements)
  int32_t out_plane_shift;  // layout of out (linear kernel without residual or query / key epilogue; 0: rows of ldo elements)
  // Readout riding on the feed-forward epilogue: token_dots[row] = sum over the features of out[row] * head_w (fp32, from
  // the rounded output), so that a mean-pooling linear head behind the layer need not read the rows again.
  const bf16_t* head_w;     // [D] or null
  float* token_dots;        // [M] (rows like out), written for the tokens the kernel stores
  float* rstd_out;          // [M]: the per-token factor of the norm in front (of the up projection; of the linear layer), or null
  bf16_t* x1_out;           // OUTP: the tokens between the two halves of the block, [M, D] rows like out; or null
  // Few-token feed-forward with the hidden units of a 32-token tile divided over `splits` workgroups (0: one): every workgroup
  // leaves its fp32 partial in split_partials [tile][splits][32 x D] and counts itself in split_counters [tile] (zero before
  // the launch); the last one to arrive adds the partials up in order, finishes the tile and sets the counter back to zero.
  int32_t splits;
  float* split_partials;
  uint32_t* split_counters;
};

// The few-token form of the projection (ffn_small.hip): packed weights, the norm in front folded into them or absent.
int norm_linear_small(const TsParams& p, int32_t K, int qk_mode, hipStream_t s, const char* name);
// The few-token form of the gated feed-forward (with_proj: the out projection in front), same conditions; 1 when the shape does
// not fit its LDS.
int swiglu_ffn_small(const TsParams& p, int32_t D, bool with_proj, bool act_folded, hipStream_t s, const char* name);

namespace {

__device__ __forceinline__ float silu_f(float v) {
  return v * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * v));
}

// Hidden unit (0..15) loaded into row slot m16 of the gate (or value) half of an up fragment: chosen so that
// accumulator register j < 8 of lane half hh holds hidden unit 8*hh + j, the k order of a W_down fragment.
__host__ __device__ __forceinline__ int up_unit_of_slot(int m16) {
  return 8 * ((m16 >> 2) & 1) + 4 * (m16 >> 3) + (m16 & 3);
}

// Constants of the gate's activation when the packed up projection carries them (see ffn_pack_piece in pack.h).
constexpr float kFoldGate = -1.4426950408889634f, kFoldValue = -0.6931471805599453f;

// ---- shared pieces ---------------------------------------------------------------------------------------------------

// Number of tokens to process: M, or *n_rows (clamped to M) when a count is given.
__device__ __forceinline__ int64_t token_count(const TsParams& p) {
  if (p.n_rows == nullptr) return p.M;
  const int64_t n = *p.n_rows;
  return n < p.M ? n : p.M;
}

// Row of x / residual / out that holds token `tok`. Tokens at or beyond the count are mapped to the last token: they
// compute bit-identical values, so loading and storing them again is benign and every wavefront issues the same
// number of memory operations.
__device__ __forceinline__ int64_t token_row(const TsParams& p, int64_t count, int64_t tok) {
  tok = tok < count ? tok : count - 1;
  return p.rows != nullptr ? static_cast<int64_t>(p.rows[tok]) : tok;
}

// Row of x that holds token `tok`: its own index when one is given, the common one otherwise.
__device__ __forceinline__ int64_t input_row(const TsParams& p, int64_t count, int64_t tok) {
  if (p.x_rows == nullptr) return token_row(p, count, tok);
  tok = tok < count ? tok : count - 1;
  return static_cast<int64_t>(p.x_rows[tok]);
}

// Rows of N tokens at once (token i = tok_of(i)), in two phases: request() issues the N index loads inside ONE test of
// the index pointer and touches none of the loaded values, row() turns entry i into a row number. Whatever the caller
// requests between the two is in flight together with the index (token_row() per token puts every load behind its own
// test of the pointer and a wait behind every load).
template <int N>
struct TokenRows {
  int64_t tok[N];
  int32_t loaded[N];
  bool indexed;
  template <typename F>
  __device__ __forceinline__ void request(const int32_t* index, int64_t count, F tok_of) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int64_t t = tok_of(i);
      tok[i] = t < count ? t : count - 1;
      loaded[i] = 0;
    }
    indexed = index != nullptr;
    if (indexed) {
#pragma unroll
      for (int i = 0; i < N; ++i) loaded[i] = index[tok[i]];
    }
  }
  // Marks the point up to which the loaded entries stay untouched (the compiler would otherwise widen them right behind
  // their loads, with a wait in front).
  __device__ __forceinline__ void arrive() {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(loaded[i]));
  }
  __device__ __forceinline__ int64_t row(int i) const { return indexed ? static_cast<int64_t>(loaded[i]) : tok[i]; }
};
template <int N, typename F>
__device__ __forceinline__ void token_rows_batch(const int32_t* index, int64_t count, F tok_of, int64_t (&row)[N]) {
  TokenRows<N> rows;
  rows.request(index, count, tok_of);
  // the entries are awaited here, on this path: left pending, the compiler protects their registers with waits for ALL
  // vector-memory operations wherever the paths of the caller meet again (in front of the MFMAs of every step)
  rows.arrive();
#pragma unroll
  for (int i = 0; i < N; ++i) row[i] = rows.row(i);
}

// Loads the wavefront's token rows as B-operand fragments: lane (l32, hh) holds features 16*ks + 8*hh .. +7 of token
// l32 of each 32-token tile.
// The same from row numbers the caller already holds (r[t]: memory row of token l32 of tile t).
template <int D, int TT>
__device__ __forceinline__ void load_token_rows_at(const TsParams& p, const int64_t (&r)[TT], int hh, bf16x8 (&xf)[TT][D / 16]) {
  constexpr int KS = D / 16;
  if (p.x_plane_shift > 0) {  // feature planes: k-step ks lies in plane (16 * ks) >> shift
    const int sh = p.x_plane_shift;
    const int64_t plane_elems = p.M << sh;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const bf16_t* row = p.x + (r[t] << sh) + hh * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        xf[t][ks] = *reinterpret_cast<const bf16x8*>(row + ((ks * 16) >> sh) * plane_elems + ((ks * 16) & ((1 << sh) - 1)));
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    const bf16_t* row = p.x + r[t] * p.ldx + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xf[t][ks] = *reinterpret_cast<const bf16x8*>(row + ks * 16);
  }
}

template <int D, int TT>
__device__ __forceinline__ void load_token_rows(const TsParams& p, int64_t count, int64_t tok0, int l32, int hh,
                                                bf16x8 (&xf)[TT][D / 16]) {
  // the row numbers of all tiles first: one memory latency in front of the row loads, not one per tile
  int64_t r[TT];
  token_rows_batch<TT>(p.x_rows != nullptr ? p.x_rows : p.rows, count, [&](int t) { return tok0 + t * 32 + l32; }, r);
  load_token_rows_at<D, TT>(p, r, hh, xf);
}

// RMS-normalises the loaded rows in place: y = bf16( x * rsqrt(mean(x^2) + eps) * w ), w read from its LDS copy.
// folded: the norm's weight is part of the layer that consumes the rows; only the per-token factor is applied.
template <int D, int TT>
__device__ __forceinline__ void normalize_tokens(float eps, const bf16_t* norm_w_lds, int hh, bf16x8 (&xf)[TT][D / 16],
                                                 bool folded = false) {
  constexpr int KS = D / 16;
  float scale[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = static_cast<float>(xf[t][ks][e]);
        ss += v * v;
      }
    ss += __shfl_xor(ss, 32, kWave);
    scale[t] = rsqrtf(ss * (1.0f / D) + eps);
  }
  // Make the packed rows opaque here: otherwise the compiler keeps all D fp32 copies from the first sweep alive for
  // the second one, which does not fit the register file next to the accumulators.
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(xf[t][ks]));
  if (folded) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
#pragma unroll
        for (int e = 0; e < 8; ++e) xf[t][ks][e] = static_cast<bf16_t>(static_cast<float>(xf[t][ks][e]) * scale[t]);
        asm volatile("" : "+v"(xf[t][ks]));
      }
    return;
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bf16x8 wv = *reinterpret_cast<const bf16x8*>(norm_w_lds + ks * 16 + hh * 8);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        xf[t][ks][e] = static_cast<bf16_t>(static_cast<float>(xf[t][ks][e]) * scale[t] * static_cast<float>(wv[e]));
      asm volatile("" : "+v"(xf[t][ks]));
    }
  }
}

// rsqrt(mean(x^2) + eps) of the loaded rows, per lane for its token of each tile; the rows themselves stay as they are
// (the norm's weight is part of the packed layer, the factor goes to the accumulators). The squares are summed two
// elements per instruction (v_dot2_f32_bf16).
template <int D, int TT>
__device__ __forceinline__ void token_rstd(float eps, const bf16x8 (&xf)[TT][D / 16], float (&rstd)[TT]) {
  typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const bf16x2 pair = {xf[t][ks][e], xf[t][ks][e + 1]};
        ss = __builtin_amdgcn_fdot2_f32_bf16(pair, pair, ss, false);
      }
    ss += __shfl_xor(ss, 32, kWave);
    rstd[t] = rsqrtf(ss * (1.0f / D) + eps);
  }
}

// Bias values of a 64-feature chunk in accumulator order: piece rb*4 + jq holds features rb*32 + jq*8 + hh*4 .. +3.
__device__ __forceinline__ void read_chunk_bias(const bf16_t* bias_lds, int hh, bf16x4 (&bv)[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) bv[q] = *reinterpret_cast<const bf16x4*>(bias_lds + (q / 4) * 32 + (q % 4) * 8 + hh * 4);
}

// The same from a float32 copy of the bias (no widening per value in the epilogue).
__device__ __forceinline__ void read_chunk_bias(const float* bias_lds, int hh, f32x4 (&bv)[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) bv[q] = *reinterpret_cast<const f32x4*>(bias_lds + (q / 4) * 32 + (q % 4) * 8 + hh * 4);
}

// Writes two 32-feature accumulator blocks (64 features) of one 32-token tile into the wavefront's epilogue tile,
// adding the bias and rounding to bf16. Accumulator register jq*4 + e of lane (l32, hh) is feature jq*8 + hh*4 + e.
template <typename BiasVec>  // bf16x4 or f32x4 pieces
__device__ __forceinline__ void tile_to_lds(uint8_t* tile, const f32x16& a0, const f32x16& a1, const BiasVec (&bv)[8],
                                            int l32, int hh, float scale = 1.0f) {
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const int col = rb * 32 + jq * 8 + hh * 4;
      bf16x4 ov;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        ov[e] = static_cast<bf16_t>(fmaf(rb == 0 ? a0[jq * 4 + e] : a1[jq * 4 + e], scale, static_cast<float>(bv[rb * 4 + jq][e])));
      *reinterpret_cast<bf16x4*>(tile + l32 * kStageRow + col * 2) = ov;
    }
  }
}

// tile_to_lds that also returns the sum of squares of the lane's 32 rounded values (half of its token's 64 features).
__device__ __forceinline__ float tile_to_lds_sumsq(uint8_t* tile, const f32x16& a0, const f32x16& a1,
                                                   const bf16x4 (&bv)[8], int l32, int hh, float scale = 1.0f) {
  float ss = 0.f;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const int col = rb * 32 + jq * 8 + hh * 4;
      bf16x4 ov;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ov[e] = static_cast<bf16_t>(fmaf(rb == 0 ? a0[jq * 4 + e] : a1[jq * 4 + e], scale, static_cast<float>(bv[rb * 4 + jq][e])));
        const float r = static_cast<float>(ov[e]);
        ss = fmaf(r, r, ss);
      }
      *reinterpret_cast<bf16x4*>(tile + l32 * kStageRow + col * 2) = ov;
    }
  }
  return ss;
}

// Sum of a value and the one held by lane ^ 32.
__device__ __forceinline__ float half_wave_pair_sum(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) + __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

}  // namespace
}  // namespace taac
