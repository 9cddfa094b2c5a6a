// Dense kernels of the token path for few tokens (gfx950, model width D = 256 or 128).
//
// The kernels of ffn.hip keep 256 or 512 tokens in a workgroup and stream the weights past them: the right shape when every
// compute unit has a tile, and a long serial walk over the weights by a handful of compute units when a batch holds a
// few thousand tokens or one request. Here the work of a 32-token tile is spread instead: the wavefronts of a workgroup share
// the tokens and divide the OUTPUT features (projection), so that each reads its own slice of the packed weights
// straight from L2 into MFMA operand registers - fragments are 1 KB of contiguous memory, no other wavefront of the workgroup
// wants them, so a stop in LDS would only add a barrier. What bounds these kernels is latency: row count -> row index ->
// token rows -> products -> store, with the weight fragments requested in front of that chain.
#include <algorithm>

#include "common.h"
#include "ts_common.h"
#include "ts_dense.h"

namespace taac {
namespace {

// Memory rows of N tokens. The index entries are requested before the number of tokens is known (the index holds M entries; what
// lies beyond the count is not used), so that the two latencies run side by side. A token at or beyond the count reads row 0:
// its values stay in its own column of every product, and it is not stored.
template <int N>
struct SmallRows {
  int64_t tok[N];
  int32_t loaded[N];
  bool indexed;
  template <typename F>
  __device__ __forceinline__ void request(const TsParams& p, const int32_t* index, F tok_of) {
    indexed = index != nullptr;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      tok[i] = tok_of(i);
      loaded[i] = 0;
    }
    if (indexed) {
#pragma unroll
      for (int i = 0; i < N; ++i) loaded[i] = index[tok[i] < p.M ? tok[i] : p.M - 1];
    }
  }
  __device__ __forceinline__ void resolve(int64_t count, int64_t (&row)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(loaded[i]));  // untouched up to here
#pragma unroll
    for (int i = 0; i < N; ++i) row[i] = tok[i] >= count ? 0 : (indexed ? static_cast<int64_t>(loaded[i]) : tok[i]);
  }
};

// [RMSNorm (weight folded) ->] linear [-> + residual], K = D, weights in fragment order. A workgroup holds the weights of D output
// features (blockIdx.y), 64 per wavefront, in registers and takes the 32-token tiles blockIdx.x, + gridDim.x, ...: the grid has no more
// workgroups than the chip has places, so that those without a tile (the number of tokens is known on the device only) do not
// stand in front of others. The rows of a tile are loaded once, contiguous pieces by neighbouring lanes, and become
// fragments in LDS. QK as in norm_linear_kernel: the features of the query
// (blockIdx.y = 0) and of the key (1) leave their sum of squares behind - as the norm's factor per token in qk_rstd when that
// is given (the workgroup holds all features of the part), per 64-feature chunk in qk_sumsq otherwise - and with QK == 2 are
// multiplied by the norm weight and rotated. Same values as norm_linear_kernel, bit for bit (same products in the same order).
// Bound by latency: count and row index -> rows -> LDS -> products -> store, 8 700 cycles of a lone workgroup; next to that a compute unit
// pulls 128 KB of weights per workgroup. q | k | v at D = 256, us, with the rows as fragments in every wavefront, the weights in
// front of them and a workgroup per tile / as it is: 512 rows 6.7 / 5.1, 8103 rows, 55 % valid 12.7 / 7.6, 16384 25.2 / 17.2; the lines are at
// dense_few_rows.
template <int D, bool RES, int QK>
__global__ __launch_bounds__(D, 2) void norm_linear_small_kernel(const TsParams p) {
  constexpr int NW = D / kNC;  // wavefronts
  constexpr int KS = D / 16;
  constexpr int NFRAG = 2 * KS;
  constexpr int kRow = D * 2 + 16;                      // bytes per row of the token tile
  constexpr int kPieces = D / 8, kStep = D / kPieces;   // 16-byte pieces of a row; rows that the threads load a piece each of
  constexpr int kPasses = 32 / kStep;
  __shared__ __attribute__((aligned(16))) uint8_t tiles[NW * kStageWave];
  __shared__ __attribute__((aligned(16))) uint8_t x_lds[2][32 * kRow];
  __shared__ __attribute__((aligned(16))) bf16_t bias_lds[NW][kNC];
  [[maybe_unused]] __shared__ float part_ss[NW][32];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int l32 = lane % 32, hh = lane / 32;
  const int nchunks = p.N / kNC;
  const int part = blockIdx.y;
  const int my_chunk = part * NW + wave;
  const bool active = my_chunk < nchunks;  // N need not be a multiple of D
  const int chunk = active ? my_chunk : nchunks - 1;
  const int piece = tid % kPieces;

  // Memory rows: of x for the pieces a thread loads; of out / residual for token 8 * i + lane / 8.
  int tok0 = static_cast<int>(blockIdx.x) * 32;
  const int stride = static_cast<int>(gridDim.x) * 32;
  const int32_t *in_index = p.x_rows != nullptr ? p.x_rows : p.rows, *out_index = p.rows;
  const int last = static_cast<int>(p.M) - 1;  // (few rows: 32 bits)
  int32_t in[kPasses], out[4];
  auto request_rows = [&](int first) {  // what lies beyond the count is not used
#pragma unroll
    for (int i = 0; i < kPasses; ++i) in[i] = first + i * kStep + tid / kPieces;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = first + i * 8 + lane / 8;
    if (in_index != nullptr) {
#pragma unroll
      for (int i = 0; i < kPasses; ++i) in[i] = in_index[in[i] < last ? in[i] : last];
    }
    if (out_index != nullptr) {
#pragma unroll
      for (int i = 0; i < 4; ++i) out[i] = out_index[out[i] < last ? out[i] : last];
    }
  };
  request_rows(tok0);
  const int count = static_cast<int>(token_count(p));
  __builtin_amdgcn_sched_barrier(0);
  // The weights depend on nothing. Half of them is in flight behind the row count and the row index, the rest behind the rows: all of
  // them in front (64 KB per wavefront group at 64 bytes a clock) would hold the rows up.
  const char* wsrc = reinterpret_cast<const char*>(p.w1) + static_cast<int64_t>(chunk) * NFRAG * kFrag;
  bf16x8 w[NFRAG];
#pragma unroll
  for (int i = 0; i < KS; ++i) w[i] = *reinterpret_cast<const bf16x8*>(wsrc + i * kFrag + lane * 16);
  __builtin_amdgcn_sched_barrier(0);
  if (tok0 >= count) return;  // whole workgroup
  bf16x8 xp[kPasses];
  auto load_rows = [&](int first) {
    int col = piece * 8;
    asm volatile("" : "+v"(col));
    const int sh = p.x_plane_shift;  // feature planes: see load_token_rows_at
    const bf16_t* base = p.x + (sh > 0 ? ((static_cast<int64_t>(col >> sh) * p.M) << sh) + (col & ((1 << sh) - 1)) : col);
    const int64_t row_stride = sh > 0 ? static_cast<int64_t>(1) << sh : p.ldx;
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      const int64_t row = first + i * kStep + tid / kPieces < count ? in[i] : 0;  // row 0 stands in beyond the count
      xp[i] = *reinterpret_cast<const bf16x8*>(base + row * row_stride);
    }
  };
  load_rows(tok0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = KS; i < NFRAG; ++i) w[i] = *reinterpret_cast<const bf16x8*>(wsrc + i * kFrag + lane * 16);
  bf16_t* bias = bias_lds[wave];
  bias[lane] = p.b1 != nullptr ? p.b1[chunk * kNC + lane] : static_cast<bf16_t>(0.f);
  uint8_t* tile = tiles + wave * kStageWave;
  const int col8 = chunk * kNC + (lane % 8) * 8;
  [[maybe_unused]] const bool qk_part = QK != 0 && chunk < p.qk_chunks;  // the same for all wavefronts of a part
  [[maybe_unused]] bf16x8 wn;
  [[maybe_unused]] bool rotate = false;
  if constexpr (QK == 2) {
#pragma unroll
    for (int e = 0; e < 8; ++e) wn[e] = static_cast<bf16_t>(1.0f);
    if (qk_part && p.qk_w != nullptr)
      wn = *reinterpret_cast<const bf16x8*>(part == 0 ? p.qk_w + col8 : p.qk_wk + (col8 - D));
    rotate = qk_part && p.cos_sin != nullptr;
  }

  for (int buf = 0; tok0 < count; tok0 += stride, buf ^= 1) {
    int32_t prow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) prow[i] = tok0 + i * 8 + lane / 8 < count ? out[i] : 0;
#pragma unroll
    for (int i = 0; i < kPasses; ++i) *reinterpret_cast<bf16x8*>(x_lds[buf] + (i * kStep + tid / kPieces) * kRow + piece * 16) = xp[i];
    bf16x8 res[4];
    if constexpr (RES) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        res[i] = *reinterpret_cast<const bf16x8*>(p.residual + static_cast<int64_t>(prow[i]) * p.ldr + chunk * kNC + (lane % 8) * 8);
    }
    __syncthreads();  // (two tiles in turn: whoever writes the next one has seen everybody leave the one before)
    f32x16 acc0, acc1;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc0[j] = acc1[j] = 0.f;
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    float rstd = 1.0f, norm_ss = 0.f;
    constexpr int kAhead = 4;  // fragments in flight (all of them do not fit next to the weights)
    auto fragment = [&](int ks) { return *reinterpret_cast<const bf16x8*>(x_lds[buf] + l32 * kRow + (ks * 16 + hh * 8) * 2); };
    bf16x8 xf[kAhead];
#pragma unroll
    for (int ks = 0; ks < kAhead; ++ks) xf[ks] = fragment(ks);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 x = xf[ks % kAhead];
      if (ks + kAhead < KS) xf[ks % kAhead] = fragment(ks + kAhead);
      acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ks], x, acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[KS + ks], x, acc1, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 8; e += 2) {  // as token_rstd
        const bf16x2 pair = {x[e], x[e + 1]};
        norm_ss = __builtin_amdgcn_fdot2_f32_bf16(pair, pair, norm_ss, false);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (p.norm_w != nullptr) {  // the norm's weight is part of the packed layer
      norm_ss += __shfl_xor(norm_ss, 32, kWave);
      rstd = rsqrtf(norm_ss * (1.0f / D) + p.eps);
    }
    if (p.rstd_out != nullptr && part == 0 && wave == 0 && hh == 0 && tok0 + l32 < count)
      p.rstd_out[token_row(p, count, tok0 + l32)] = rstd;

    bf16x4 bv[8];
    read_chunk_bias(bias, hh, bv);
    if constexpr (QK != 0) {
      if (qk_part && (p.qk_sumsq != nullptr || p.qk_rstd != nullptr)) {
        const float ss = half_wave_pair_sum(tile_to_lds_sumsq(tile, acc0, acc1, bv, l32, hh, rstd));
        if (p.qk_rstd != nullptr) {
          if (hh == 0) part_ss[wave][l32] = ss;
          __syncthreads();
          if (wave == 0 && hh == 0) {
            float total = 0.f;
#pragma unroll
            for (int c = 0; c < NW; ++c) total += part_ss[c][l32];
            const int64_t tok = tok0 + l32;
            const int64_t row = token_row(p, count, tok);
            if (tok < count) p.qk_rstd[part * p.M + row] = rsqrtf(total * (1.0f / D) + p.qk_eps);
          }
        } else {
          const int64_t row = token_row(p, count, tok0 + l32);
          if (hh == 0 && tok0 + l32 < count) p.qk_sumsq[static_cast<int64_t>(chunk) * p.M + row] = ss;
        }
      } else {
        tile_to_lds(tile, acc0, acc1, bv, l32, hh, rstd);
      }
    } else {
      tile_to_lds(tile, acc0, acc1, bv, l32, hh, rstd);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (active) {
      int col = col8;
      asm volatile("" : "+v"(col));  // (addresses formed ahead of the loop would be spilled)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = i * 8 + lane / 8;
        bf16x8 v = *reinterpret_cast<const bf16x8*>(tile + row * kStageRow + (lane % 8) * 16);
        if constexpr (RES) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) + static_cast<float>(res[i][e]));
        }
        if constexpr (QK == 2) {
          if (qk_part) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = static_cast<float>(v[e]) * static_cast<float>(wn[e]);
            if (rotate) {
              const int pos = static_cast<int>(input_row(p, count, tok0 + row) % p.tokens_per_sample);
              const bf16x8 cs = *reinterpret_cast<const bf16x8*>(p.cos_sin + static_cast<int64_t>(pos) * p.head_dim + col % p.head_dim);
#pragma unroll
              for (int e = 0; e < 8; e += 2) {
                const float even = f[e], odd = f[e + 1];
                const float cv = static_cast<float>(cs[e]), sv = static_cast<float>(cs[e + 1]);
                f[e] = even * cv - odd * sv;
                f[e + 1] = even * sv + odd * cv;
              }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(f[e]);
          }
        }
        if (tok0 + row >= count) continue;
        // feature planes: column c lies in plane c >> shift, at c % 2^shift of the row
        const int64_t at = p.out_plane_shift > 0
                               ? (((static_cast<int64_t>(col >> p.out_plane_shift) * p.M + prow[i]) << p.out_plane_shift) +
                                  (col & ((1 << p.out_plane_shift) - 1)))
                               : static_cast<int64_t>(prow[i]) * p.ldo + col;
        *reinterpret_cast<bf16x8*>(p.out + at) = v;
      }
    }
    // (not a tile ahead: next to the weights there are no registers for the rows, and reloads of spilled ones wait for all loads)
    if (tok0 + stride < count) {
      request_rows(tok0 + stride);
      load_rows(tok0 + stride);
    }
  }
}

// Data that other workgroups of the same launch read: accesses at the scope of the whole chip, which go through the L2 of the die
// to the memory all dies share. (Ordinary stores with a fence behind them write back and drop everything the die's L2 holds:
// 8 us per launch.)
// Sixteen bytes per lane and access: as atomic accesses, eight bytes at most, twice as many requests leave the compute unit (eight
// partials of 32 KB: 2.7 us more).
// Ordering is the caller's: a wait and a barrier in front of the count that publishes the stores, a barrier behind it for the loads.
constexpr int kThroughL2 = 16;  // the sc1 bit of a buffer access: coherent at the scope of the chip
struct SharedPartials {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ SharedPartials(float* base, int bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000)) {}
  __device__ __forceinline__ void store(int at, const f32x4& v) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, at, 0, kThroughL2);
  }
  __device__ __forceinline__ f32x4 load(int at) const {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, kThroughL2));
  }
};

// ------------------------------------------------------------------------------------------------------------------
// The feed-forward half for few tokens: [out projection + residual ->] RMSNorm -> up -> SiLU-gate -> down -> + residual of
// 32 or 64 tokens per workgroup (the products, blobs and roundings of swiglu_ffn_kernel). The wavefronts, one per 32 features, share
// the tokens. The projection and the down projection are divided by OUTPUT features, the up projection by HIDDEN units; the
// normalised tokens and the hidden state, as operand fragments, meet in LDS. (With the down projection divided by hidden units, too,
// every wavefront holds a partial of all features: four times the accumulators, 128 KB of partials through LDS, and one wavefront
// per SIMD, whose instructions then stand between its products.)
//
// A wavefront's weights are one stream of fragments, L2 -> registers, through a ring of KS fragments (16 KB in flight at
// D = 256, 128 KB per workgroup): projection, then the up fragments of its 16-unit chunks, then the down fragments of its
// features; a slot is requested again as soon as its product is issued.
// Bound, one tile: the weights a compute unit pulls from L2 at 64 bytes a clock (1.6 MB at D = 256, F = 1024: 24 000 of the kernel's
// 38 000 cycles; the rest is the chain row index -> rows -> projection -> norm in front, and the stores). Two tiles halve that and are
// bound by the products and the activation, which add: 1.7 us per 1000 tokens at D = 256, F = 1024.
// One launch, us, this form / the one with partials of all features: D = 256, F = 1024 - 4096 rows 19.9 / 25.1, 8103 rows 23.0 /
// 27.8, 16384 rows 32.4 / 53.8, 9648 rows, 6100 valid 20.4 / 26.9; F = 512 - 8103 rows 15.1 / 18.8; D = 128, F = 512 - 512 rows 8.2 / 9.2.
// splits > 1 (see TsParams): for batches that leave most of the chip idle even so, the hidden units of a tile are also divided over
// workgroups; the exchange costs 4 - 5 us, and the rule is at ffn_splits.
// ------------------------------------------------------------------------------------------------------------------
constexpr int kPiece = 64;  // 16-unit chunks whose hidden state lies in LDS in one piece at most (F = 1024)

// LDS of the kernel for workgroups of TT token tiles and `chunks` chunks of hidden units, at most `slab` at a time: first the normalised
// rows of a tile that are kept (one tile: read once, but the hidden state need not wait for it; two tiles, D = 256: the second one's
// fragments, for which there are no registers), then the tokens as they come in (and the other normalised rows), whose place the hidden
// state takes. The biases and sums come behind.
__host__ __device__ constexpr int small_kept_bytes(int D, int TT) { return TT == 1 || D == 256 ? 32 * (D * 2 + 16) : 0; }
__host__ __device__ constexpr int small_tile_bytes(int D, int TT, int chunks, int slab) {
  const int rows = 32 * (D * 2 + 16), hidden = TT * (chunks < slab ? chunks : slab) * kFrag;
  const int tokens = 2 * TT * rows - small_kept_bytes(D, TT);
  return small_kept_bytes(D, TT) + (hidden > tokens ? hidden : tokens);
}

// Groups of one chunk per wavefront that a workgroup of the kernel takes at most.
__host__ __device__ constexpr int small_groups(int D, int F, int splits) {
  return ((F / kHU + D / 32 - 1) / (D / 32) + splits - 1) / splits;
}

// What a workgroup asks for before it knows the number of tokens: the row index of its tiles and the projection's weights.
template <int D, int TT>
struct SmallTokens {
  static constexpr int kPieces = D / 8;                             // 16-byte pieces of a row
  static constexpr int kStep = D / 32 * kWave / kPieces;            // rows that the threads load a piece each of
  static constexpr int kPasses = 32 * TT / kStep;
  SmallRows<kPasses> in;  // rows of x, by pieces
  SmallRows<TT> out;      // rows of residual / out: token l32 of each tile
  __device__ __forceinline__ void request(const TsParams& p, int64_t tok0, int tid, int l32) {
    in.request(p, p.x_rows != nullptr ? p.x_rows : p.rows, [&](int i) { return tok0 + i * kStep + tid / kPieces; });
    out.request(p, p.rows, [&](int t) { return tok0 + t * 32 + l32; });
  }
};

template <int D, int TT, bool OUTP, bool FOLD, int SLAB>
__device__ __forceinline__ void ffn_small_tile(const TsParams& p, uint8_t* smem, int64_t count, int tile, int split,
                                               SmallTokens<D, TT>& tokens, bf16x8 (&ring)[D / 16]) {
  constexpr int KS = D / 16, MB = D / 32;
  constexpr int NW = MB;                      // wavefronts
  constexpr int CFRAG = KS + MB;
  constexpr int kRow = D * 2 + 16;            // bytes per row of a token tile
  constexpr int kPart = MB * 4 * kWave * 16;  // bytes of one split's partial
  constexpr int XT = D == 256 ? 1 : TT;       // tiles whose normalised tokens stay in registers
  constexpr int kKept = small_kept_bytes(D, TT);
  static_assert(KS == 2 * NW, "a ring holds the down fragments of two groups of chunks");
  constexpr bool SLABS = SLAB > 0;
  const int F = p.F;
  const int nchunks = F / kHU;
  const int splits = TT == 1 && p.splits > 1 ? p.splits : 1;
  const int shift = __builtin_ctz(splits);  // a power of two (ffn_splits)
  const int groups = ((nchunks + NW - 1) / NW + splits - 1) >> shift;
  // normalised rows of a tile; rows as they come in, then between the halves; hidden state
  auto normed_lds = [&](int t) {
    if constexpr (TT == 1) return smem;
    if (kKept > 0) return t == 1 ? smem : smem + kKept;
    return smem + t * 32 * kRow;
  };
  uint8_t* x_lds = smem + (TT == 1 ? kKept : kKept + (kKept > 0 ? 1 : 2) * 32 * kRow);
  uint8_t* hidden_lds = smem + kKept;
  float* bias_lds = reinterpret_cast<float*>(smem + small_tile_bytes(D, TT, groups * NW, SLABS ? SLAB : kPiece));
  bf16_t* end_lds = reinterpret_cast<bf16_t*>(bias_lds + 2 * F);  // down-projection bias, readout weight
  float* sums = reinterpret_cast<float*>(end_lds + 2 * D);  // [TT][NW][32]

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int l32 = lane % 32, hh = lane / 32;
  const int lane16 = lane * 16;
  const int64_t tok0 = static_cast<int64_t>(tile) * (32 * TT);

  // Weights: buffer accesses, whose address is a lane offset, a scalar offset and a constant (no vector arithmetic per load).
  // Group k of the workgroup holds the NW chunks from (k * splits + split) * NW on, the wavefront's own one at + wave.
  const int blob_bytes = nchunks * CFRAG * kFrag;
  const auto blob = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w1), 0, blob_bytes, 0x00020000);
  auto request = [&](int at, int constant) {
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(blob, lane16 + constant, at, 0));
  };
  auto first_chunk = [&](int group) { return ((group << shift) + split) * NW; };
  auto own_chunk = [&](int group) {
    const int chunk = first_chunk(group) + wave;
    return chunk < nchunks ? chunk : nchunks - 1;
  };
  auto up_at = [&](int group) { return own_chunk(group) * (CFRAG * kFrag); };
  const int blob_end = blob_bytes - kFrag;  // (the last fragment stands in for those that are requested and not used)
  auto request_up = [&](int at, auto ic) {
    constexpr int i = decltype(ic)::value;
    return request(at + i / 4 * (4 * kFrag), i % 4 * kFrag);
  };
  auto request_down = [&](int group, int j) {
    const int at = (first_chunk(group) + j) * (CFRAG * kFrag) + (KS + wave) * kFrag;
    return request(at < blob_end ? at : blob_end, 0);
  };
  int64_t xrow[SmallTokens<D, TT>::kPasses], row[TT];  // row: of token l32 of a tile in residual / out
  tokens.in.resolve(count, xrow);
  tokens.out.resolve(count, row);
  // The token rows are loaded once per workgroup, contiguous pieces by neighbouring lanes (as operand fragments by every wavefront,
  // 32 bytes of 32 rows an access, they cost the compute unit 16 times the requests), and become fragments in LDS.
  constexpr int kPasses = SmallTokens<D, TT>::kPasses, kStep = SmallTokens<D, TT>::kStep, kPieces = SmallTokens<D, TT>::kPieces;
  const int piece = tid % kPieces;
  bf16x8 xp[kPasses];
  {
    const int col = piece * 8;
    const int sh = p.x_plane_shift;
    const bf16_t* base = p.x + (sh > 0 ? ((static_cast<int64_t>(col >> sh) * p.M) << sh) + (col & ((1 << sh) - 1)) : col);
    const int64_t stride = sh > 0 ? static_cast<int64_t>(1) << sh : p.ldx;
#pragma unroll
    for (int i = 0; i < kPasses; ++i) xp[i] = *reinterpret_cast<const bf16x8*>(base + xrow[i] * stride);
  }
  // Four features per register quad of the lane's block, in accumulator order. A vector that is absent is read from the weights
  // instead (finite, in bounds for D values) and cleared where it is used: no branch between the loads.
  auto feature_vectors = [&](const bf16_t* v, bf16x4 (&dst)[4]) {
    const bf16_t* src = v != nullptr ? v : p.w1;
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) dst[jq] = *reinterpret_cast<const bf16x4*>(src + wave * 32 + jq * 8 + hh * 4);
  };
  [[maybe_unused]] bf16x4 hv[TT][4], b0v[4];  // block input (then x1, in accumulator order), projection bias
  auto block_input = [&]() {
    if constexpr (OUTP) {
#pragma unroll
      for (int t = 0; t < TT; ++t) feature_vectors(p.residual + row[t] * p.ldr, hv[t]);
      feature_vectors(p.b0, b0v);
    }
  };
  if constexpr (TT == 1) block_input();
  // first-layer bias, gated half first; FOLD: with the constants the packed layer carries. 8 entries per thread and round.
  auto bias_piece = [&](int i) {
    const bool gated = i < F;  // F is a multiple of 32: a piece lies in one half
    return *reinterpret_cast<const bf16x8*>(p.b1 != nullptr ? p.b1 + (gated == (p.gate_first != 0) ? i % F : F + i % F) : p.w1);
  };
  auto store_bias = [&](int i, bf16x8 v) {
    const float c = p.b1 == nullptr ? 0.f : (!FOLD ? 1.f : (i < F ? kFoldGate : kFoldValue));
    f32x4 lo, hi;  // widened once, here, not per chunk
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] = static_cast<float>(static_cast<bf16_t>(static_cast<float>(v[e]) * c));
      hi[e] = static_cast<float>(static_cast<bf16_t>(static_cast<float>(v[4 + e]) * c));
    }
    if (i < 2 * F) {
      *reinterpret_cast<f32x4*>(bias_lds + i) = lo;
      *reinterpret_cast<f32x4*>(bias_lds + i + 4) = hi;
    }
  };
  const bf16x8 bias_regs = bias_piece(tid * 8 < 2 * F ? tid * 8 : 0);
  const bf16_t* end_src = tid < D / 8 ? p.b2 : p.head_w;
  bf16x8 end_regs = *reinterpret_cast<const bf16x8*>((end_src != nullptr ? end_src : p.w1) + tid % (D / 8) * 8);
  __builtin_amdgcn_sched_barrier(0);
  // Groups in which the wavefront has a chunk: all but perhaps the last one of the workgroup. (A wavefront without a chunk in a slab
  // goes through the motions with the last chunk: what it leaves in its place of the hidden state is not used.)
  const int all_own = first_chunk(groups - 1) + wave < nchunks ? groups : groups - 1;
  constexpr int kSlabGroups = (SLABS ? SLAB : kPiece) / NW;
  auto ring_up = [&](int group) {
    const int at = up_at(group);
    static_for<KS>([&](auto ic) { ring[decltype(ic)::value] = request_up(at, ic); });
  };
  if constexpr (!OUTP) ring_up(0);
#pragma unroll
  for (int i = 0; i < kPasses; ++i) *reinterpret_cast<bf16x8*>(x_lds + (i * kStep + tid / kPieces) * kRow + piece * 16) = xp[i];
  if constexpr (TT > 1) {  // (no registers for it next to the rows)
    __builtin_amdgcn_sched_barrier(0);
    block_input();
  }
  __syncthreads();
  auto fragment = [&](const uint8_t* rows, int ks) {
    return *reinterpret_cast<const bf16x8*>(rows + l32 * kRow + (ks * 16 + hh * 8) * 2);
  };
  bf16x8 xf[XT][KS];
#pragma unroll
  for (int t = 0; t < XT; ++t)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xf[t][ks] = fragment(x_lds + t * 32 * kRow, ks);
  // Fragment ks of tile t: from the registers, or read from `far`, two products ahead.
  auto products = [&](f32x16 (&acc)[TT], const uint8_t* far, auto reload) {
    bf16x8 ahead[2];
    if constexpr (XT < TT) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) ahead[ks] = fragment(far, ks);
    }
    static_for<KS>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
#pragma unroll
      for (int t = 0; t < XT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i], xf[t][i], acc[t], 0, 0, 0);
      if constexpr (XT < TT) {
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i], ahead[i % 2], acc[1], 0, 0, 0);
        if constexpr (i + 2 < KS) ahead[i % 2] = fragment(far, i + 2);
      }
      reload(ic);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  if constexpr (OUTP) {
    const float b0_on = p.b0 != nullptr ? 1.f : 0.f;
    f32x16 acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;
    const int at = up_at(0);
    products(acc, x_lds + 32 * kRow, [&](auto ic) { ring[decltype(ic)::value] = request_up(at, ic); });
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      float ss = 0.f;
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        bf16x4 x1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lin = static_cast<float>(static_cast<bf16_t>(fmaf(static_cast<float>(b0v[jq][e]), b0_on, acc[t][jq * 4 + e])));
          x1[e] = static_cast<bf16_t>(lin + static_cast<float>(hv[t][jq][e]));
          const float r = static_cast<float>(x1[e]);
          ss = fmaf(r, r, ss);
        }
        hv[t][jq] = x1;
      }
      ss = half_wave_pair_sum(ss);
      if (hh == 0) sums[(t * NW + wave) * 32 + l32] = ss;
    }
  }
  store_bias(tid * 8, bias_regs);
  for (int i = (NW * kWave + tid) * 8; i < 2 * F; i += NW * kWave * 8) store_bias(i, bias_piece(i));
  if (tid < 2 * (D / 8)) {
    if (end_src == nullptr) {
#pragma unroll
      for (int e = 0; e < 8; ++e) end_regs[e] = static_cast<bf16_t>(0.f);
    }
    *reinterpret_cast<bf16x8*>(end_lds + tid * 8) = end_regs;
  }
  if constexpr (OUTP) {
    __syncthreads();
    const bool keep = p.x1_out != nullptr && split == 0;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += sums[(t * NW + w) * 32 + l32];
      const float scale = p.norm_w != nullptr ? rsqrtf(sum * (1.0f / D) + p.eps) : 1.0f;
      if (p.rstd_out != nullptr && split == 0 && wave == 0 && hh == 0 && tok0 + t * 32 + l32 < count) p.rstd_out[row[t]] = scale;
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {  // every wavefront normalises the features it has projected
        const int at = l32 * kRow + (wave * 32 + jq * 8 + hh * 4) * 2;
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(hv[t][jq][e]) * scale);
        *reinterpret_cast<bf16x4*>(normed_lds(t) + at) = v;
        if (keep) *reinterpret_cast<bf16x4*>(x_lds + t * 32 * kRow + at) = hv[t][jq];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < XT; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) xf[t][ks] = fragment(normed_lds(t), ks);
    if (keep) {
#pragma unroll
      for (int i = 0; i < kPasses; ++i) {
        const int t = i * kStep + tid / kPieces;
        if (tok0 + t >= count) continue;
        const int64_t r = p.rows != nullptr ? static_cast<int64_t>(p.rows[tok0 + t]) : tok0 + t;
        *reinterpret_cast<bf16x8*>(p.x1_out + r * D + piece * 8) = *reinterpret_cast<const bf16x8*>(x_lds + t * kRow + piece * 16);
      }
      if constexpr (TT == 1) __syncthreads();  // the hidden state takes the place of x1
    }
  } else {
    // the rows are whole in every wavefront; the second tile's, where it stays in LDS, is normalised by the first
    if constexpr (XT < TT) {
      if (wave == 0) {
        bf16x8 far[1][KS];
        float rstd[1] = {1.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) far[0][ks] = fragment(x_lds + 32 * kRow, ks);
        if (p.norm_w != nullptr) token_rstd<D, 1>(p.eps, far, rstd);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
          for (int e = 0; e < 8; ++e) far[0][ks][e] = static_cast<bf16_t>(static_cast<float>(far[0][ks][e]) * rstd[0]);
          *reinterpret_cast<bf16x8*>(normed_lds(1) + l32 * kRow + (ks * 16 + hh * 8) * 2) = far[0][ks];
        }
      }
    }
    if (p.norm_w != nullptr) {
      float rstd[XT];
      token_rstd<D, XT>(p.eps, xf, rstd);
#pragma unroll
      for (int t = 0; t < XT; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int e = 0; e < 8; ++e) xf[t][ks][e] = static_cast<bf16_t>(static_cast<float>(xf[t][ks][e]) * rstd[t]);
    }
    if constexpr (TT == 1) __syncthreads();  // as below, and the biases
  }
  if constexpr (TT > 1) __syncthreads();  // the hidden state takes the place of the tokens
  if constexpr (OUTP && SLABS) {  // x1 is kept as it is rounded (widened ahead of the loop it would be spilled)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) asm volatile("" : "+v"(hv[t][jq]));
  }

  f32x16 total[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) total[t][j] = 0.f;
  for (int slab = 0; slab < (SLABS ? groups : 1); slab += kSlabGroups) {
    const int slab_end = SLABS && slab + kSlabGroups < groups ? slab + kSlabGroups : groups;
    const int own_end = slab_end < all_own ? slab_end : all_own;
    auto up_chunk = [&](int group, auto last_c) {
      constexpr bool last = decltype(last_c)::value;
      const int unit = own_chunk(group) * kHU + hh * 8;
      const int next = up_at(group + 1);
      f32x16 gu[TT];
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 b = *reinterpret_cast<const f32x4*>(bias_lds + (q < 2 ? 0 : F) + unit + q % 2 * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) gu[t][q * 4 + e] = b[e];
        }
      products(gu, normed_lds(TT - 1), [&](auto ic) {
        constexpr int i = decltype(ic)::value;
        ring[i] = last ? request_down(slab + i / NW, i % NW) : request_up(next, ic);
      });
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        bf16x8 hb;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if constexpr (FOLD)
            hb[e] = static_cast<bf16_t>(gu[t][e] * gu[t][8 + e] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gu[t][e])));
          else
            hb[e] = static_cast<bf16_t>(silu_f(gu[t][e]) * gu[t][8 + e]);
        }
        *reinterpret_cast<bf16x8*>(hidden_lds + (((group - slab) * NW + wave) * TT + t) * kFrag + lane16) = hb;
      }
    };
    for (int group = slab; group + 1 < own_end; ++group) up_chunk(group, std::false_type{});
    up_chunk(own_end > slab ? own_end - 1 : slab, std::true_type{});
    __syncthreads();
    // two groups a round; only the last group of a workgroup may be a partial one
    auto down_groups = [&](int group, auto last_c) {
      constexpr bool last = decltype(last_c)::value;
      static_for<KS / 4>([&](auto quad_c) {
        constexpr int q = decltype(quad_c)::value;
        const int g = group + q * 4 / NW;
        if (last && g >= slab_end) return;
        bf16x8 hb[4][TT];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < TT; ++t)
            hb[j][t] = *reinterpret_cast<const bf16x8*>(hidden_lds + (((group - slab) * NW + q * 4 + j) * TT + t) * kFrag + lane16);
        static_for<4>([&](auto jc) {
          constexpr int j = decltype(jc)::value, i = q * 4 + j;
          if (!last || first_chunk(g) + i % NW < nchunks) {
#pragma unroll
            for (int t = 0; t < TT; ++t) total[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i], hb[j][t], total[t], 0, 0, 0);
          }
          if constexpr (!last) ring[i] = request_down(g + 2, i % NW);
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    };
    int group = slab;
    for (; group + 2 < slab_end; group += 2) down_groups(group, std::false_type{});
    down_groups(group, std::true_type{});
    if constexpr (SLABS) {
      if (slab_end < groups) {  // the ring starts anew
        ring_up(slab_end);
        __syncthreads();  // the hidden state of this slab has been read
      }
    }
  }

  if (TT == 1 && splits > 1) {
    // The partial of this workgroup becomes visible to the chip, then the workgroup counts itself: whoever counts last finds all
    // partials of the tile (nobody waits for anybody). They are added in the order of the splits: the same result every run.
    const SharedPartials parts(p.split_partials + static_cast<int64_t>(tile) * splits * (kPart / 4), splits * kPart);
    const int lane_at = wave * (4 * kWave * 16) + lane16;  // of a partial: [feature block][register quad][lane]
    const int at = split * kPart + lane_at;
#pragma unroll
    for (int jq = 0; jq < 4; ++jq)
      parts.store(at + jq * (kWave * 16), f32x4{total[0][jq * 4], total[0][jq * 4 + 1], total[0][jq * 4 + 2], total[0][jq * 4 + 3]});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's partials have reached the chip's common memory
    __syncthreads();
    uint32_t* arrived = reinterpret_cast<uint32_t*>(sums);
    if (tid == 0)
      *arrived = __hip_atomic_fetch_add(p.split_counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const bool last = *arrived == static_cast<uint32_t>(splits - 1);
    __syncthreads();  // (the row sums of the readout reuse the word)
    if (!last) return;
    if (tid == 0) p.split_counters[tile] = 0u;
#pragma unroll
    for (int j = 0; j < 16; ++j) total[0][j] = 0.f;
    auto add_partials = [&](auto number) {  // all in flight at once
      constexpr int n = decltype(number)::value;
      f32x4 v[n][4];
#pragma unroll
      for (int u = 0; u < n; ++u)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) v[u][jq] = parts.load(u * kPart + lane_at + jq * (kWave * 16));
#pragma unroll
      for (int u = 0; u < n; ++u)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq)
#pragma unroll
          for (int e = 0; e < 4; ++e) total[0][jq * 4 + e] += v[u][jq][e];
    };
    if (splits == 2)  // 2 or 4 (ffn_splits)
      add_partials(std::integral_constant<int, 2>{});
    else
      add_partials(std::integral_constant<int, 4>{});
  }
  bf16x4 result[TT][4];
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    float hdot = 0.f;
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const int col = wave * 32 + jq * 8 + hh * 4;
      const bf16x4 b2v = *reinterpret_cast<const bf16x4*>(end_lds + col), hwv = *reinterpret_cast<const bf16x4*>(end_lds + D + col);
      f32x4 s;
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = total[t][jq * 4 + e] + static_cast<float>(b2v[e]);
      bf16x4 o;
      if constexpr (OUTP) {  // x1 + down, rounded once
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16_t>(s[e] + static_cast<float>(hv[t][jq][e]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16_t>(s[e]);
        if (p.residual != nullptr) {
          const bf16x4 r = *reinterpret_cast<const bf16x4*>(p.residual + row[t] * p.ldr + col);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16_t>(static_cast<float>(o[e]) + static_cast<float>(r[e]));
        }
      }
      result[t][jq] = o;
#pragma unroll
      for (int e = 0; e < 4; ++e) hdot = fmaf(static_cast<float>(o[e]), static_cast<float>(hwv[e]), hdot);
    }
    if (p.head_w != nullptr) {
      hdot = half_wave_pair_sum(hdot);
      if (hh == 0) sums[(t * NW + wave) * 32 + l32] = hdot;
    }
  }
  if (p.head_w != nullptr) {  // (in front of the stores: the barrier would wait for them)
    __syncthreads();
    if (wave < TT && hh == 0 && tok0 + wave * 32 + l32 < count) {
      float d = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) d += sums[(wave * NW + w) * 32 + l32];
      p.token_dots[TT == 1 || wave == 0 ? row[0] : row[TT - 1]] = d;
    }
  }
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    if (tok0 + t * 32 + l32 >= count) continue;
#pragma unroll
    for (int jq = 0; jq < 4; ++jq)
      *reinterpret_cast<bf16x4*>(p.out + row[t] * p.ldo + wave * 32 + jq * 8 + hh * 4) = result[t][jq];
  }
}

// Forms of the kernel. One tile per workgroup: its hidden state in one piece / in slabs of 1024 units / (D = 128) of 512, whose smaller
// LDS leaves a compute unit three workgroups instead of two or one. For more rows than the chip has places for one-tile workgroups: the
// number of tokens, known on the device only, decides whether workgroups take one tile or two (D = 256, F = 1024: 12288 rows, all valid,
// 28.0 us, 39.3 with one tile in two rounds; 6758 valid 21.2, one tile in one round), in one piece / in slabs of 512 units (D = 128: 384 for
// two tiles) where F is over 1024 or the pieces would leave a compute unit fewer workgroups. One launch behind the out projection, us, with
// slabs for one tile only and places that do not depend on F / as it is: D = 256, F = 2048 - 9216 rows 66 / 45, 16384 78 / 61, 55 % valid 65 / 42,
// 24576 117 / 98 and 68 / 51 (12288 rows, 55 % valid, 34 / 36: one tile in the larger kernel); D = 128 - F = 640, 40960 rows 40 / 34 and 27 / 21; F =
// 1024, 16384 rows 24.4 / 21.9 and 23.0 / 18.9, 32768 38 / 34 and 36 / 27; F = 2048, 24576 rows 65 / 52 and 40 / 35, 49152 121 / 86 and 75 / 51.
enum { kSmallOne, kSmallSlabs, kSmallHalfSlabs, kSmallPair, kSmallPairSlabs };
__host__ __device__ constexpr bool small_pairs(int form) { return form == kSmallPair || form == kSmallPairSlabs; }
// Chunks of hidden units in a slab of workgroups of TT tiles, 0 where they lie in one piece.
__host__ __device__ constexpr int small_slab(int D, int TT, int form) {
  if (form == kSmallOne || form == kSmallPair) return 0;
  if (form == kSmallSlabs) return kPiece;
  return TT == 2 ? (D == 256 ? 32 : 24) : (D == 256 ? kPiece : 32);
}

template <int D, bool OUTP, bool FOLD, int FORM>
__global__ __launch_bounds__(D / 32 * kWave, D == 256 || small_pairs(FORM) ? 2 : 3) void swiglu_ffn_small_kernel(const TsParams p) {
  constexpr int KS = D / 16;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  // Workgroup i runs on die i % 8: with two or four splits a die reads only its own share of the hidden units' weights.
  const int shift = __builtin_ctz(p.splits > 1 ? p.splits : 1);
  const int tile = static_cast<int>(blockIdx.x) >> shift, split = static_cast<int>(blockIdx.x) & ((1 << shift) - 1);
  // Requests in the order in which their values are needed (they arrive in that order): row index and count, the projection's
  // weights behind them, then - one latency later - the token rows, and what is used after the projection.
  SmallTokens<D, 1> one;
  [[maybe_unused]] SmallTokens<D, 2> two;
  one.request(p, static_cast<int64_t>(tile) * 32, tid, lane % 32);
  if constexpr (FORM == kSmallPair) two.request(p, static_cast<int64_t>(tile) * 64, tid, lane % 32);
  const int64_t count = token_count(p);
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 ring[KS];
  if constexpr (OUTP) {
    const auto w0 = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w0), 0, D * D * 2, 0x00020000);
    static_for<KS>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      ring[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(w0, lane * 16 + i % 4 * kFrag,
                                                                                 wave * (KS * kFrag) + i / 4 * (4 * kFrag), 0));
    });
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (small_pairs(FORM)) {
    if (count > static_cast<int64_t>(p.units) * 32) {  // p.units: workgroups that run at once
      if constexpr (FORM == kSmallPairSlabs) two.request(p, static_cast<int64_t>(tile) * 64, tid, lane % 32);
      if (static_cast<int64_t>(tile) * 64 < count) ffn_small_tile<D, 2, OUTP, FOLD, small_slab(D, 2, FORM)>(p, smem, count, tile, 0, two, ring);
      return;
    }
  }
  if (static_cast<int64_t>(tile) * 32 < count)
    ffn_small_tile<D, 1, OUTP, FOLD, small_slab(D, 1, FORM)>(p, smem, count, tile, split, one, ring);
}

}  // namespace

// Two or four workgroups per token tile as long as the tiles leave them a compute unit each, every wavefront keeps two chunks of
// hidden units, and the weights are worth the exchange. Whole 4-block calls, 1 / 2 / 4 / 8 splits, us: D = 256, F = 1024 - 1 x 512
// positions 146 / 125 / 116 / 119, 8 x 256 139 / 121 / 119; F = 512 (two chunks at two splits) - 1 x 512 115 / 112 / 108, 4 x 512
// 116 / 115 / 116; D = 128, F = 512 - 1 x 512 86 / 84 / 82, 8 x 256 81 / 80 / 80; F = 256 - 78 / 79 / 79, 74 / 75 / 77. (Those of a kernel whose
// exchange was of all features, which gained from eight at F = 2048, 161 -> 156; four in this one: 130.)
int ffn_splits(int64_t M, int32_t D, int32_t F) {
  const int64_t tiles = (M + 31) / 32;
  const int cus = compute_units();
  int splits = 1;
  if (ffn_few_rows(M, D, F) && F >= 512)
    while (splits < 4 && 2 * splits * tiles <= cus && 2 * splits * 2 * (D / 32) * kHU <= F) splits *= 2;
  return splits;
}

int64_t ffn_split_bytes(int64_t M, int32_t D, int32_t F) {
  const int splits = ffn_splits(M, D, F);
  if (splits == 1) return 0;
  const int64_t tiles = (M + 31) / 32;
  return tiles * splits * 32 * D * 4 + (tiles * 4 + 255) / 256 * 256;
}

int norm_linear_small(const TsParams& p, int32_t K, int qk_mode, hipStream_t s, const char* name) {
  // Places for workgroups: two per compute unit at K = 256 (registers), six at 128.
  const int64_t tiles = (p.M + 31) / 32, parts = (p.N + K - 1) / K, places = static_cast<int64_t>(compute_units()) * (K == 256 ? 2 : 6);
  const int64_t columns = places / parts > 0 ? places / parts : 1;
  const dim3 grid(static_cast<uint32_t>(tiles < columns ? tiles : columns), static_cast<uint32_t>(parts));
#define TAAC_SMALL(KK, RR, QQ)                                                                    \
  do {                                                                                            \
    hipLaunchKernelGGL((norm_linear_small_kernel<KK, RR, QQ>), grid, dim3(KK), 0, s, p);          \
    return check_launch(name);                                                                    \
  } while (0)
  if (K == 256) {
    if (qk_mode == 2) TAAC_SMALL(256, false, 2);
    if (qk_mode == 1) TAAC_SMALL(256, false, 1);
    if (p.residual != nullptr) TAAC_SMALL(256, true, 0);
    TAAC_SMALL(256, false, 0);
  }
  if (qk_mode == 2) TAAC_SMALL(128, false, 2);
  if (qk_mode == 1) TAAC_SMALL(128, false, 1);
  if (p.residual != nullptr) TAAC_SMALL(128, true, 0);
  TAAC_SMALL(128, false, 0);
#undef TAAC_SMALL
}

// Bytes of LDS of a form (of the larger of the tiles its workgroups may take), and workgroups of it that a compute unit holds: by its
// registers (launch bounds) and by its LDS, which is handed out in pieces of 1280 bytes.
namespace {
int small_lds(int D, int F, int chunks, int form) {
  const int tt = small_pairs(form) ? 2 : 1;
  auto tile = [&](int of) { return small_tile_bytes(D, of, chunks, small_slab(D, of, form) > 0 ? small_slab(D, of, form) : kPiece); };
  const int tile_bytes = tt == 2 ? std::max(tile(1), tile(2)) : tile(1);
  return tile_bytes + 2 * F * 4 + 4 * D + tt * (D / 32) * 32 * 4;
}
int small_places(int D, int F, int chunks, int form) {
  const int by_registers = D == 256 ? 1 : (small_pairs(form) ? 2 : 3);
  return std::min(by_registers, kMaxLdsBytes / ((small_lds(D, F, chunks, form) + 1279) / 1280 * 1280));
}

}  // namespace

int swiglu_ffn_small(const TsParams& params, int32_t D, bool with_proj, bool act_folded, hipStream_t s, const char* name) {
  TsParams p = params;
  const int splits = p.splits > 1 ? p.splits : 1;
  const int64_t tiles = (p.M + 31) / 32;
  const int chunks = small_groups(D, p.F, splits) * (D / 32);
  auto places = [&](int form) { return small_places(D, p.F, chunks, form) * p.units; };
  auto in_one_round = [&](int form) { return tiles * splits <= places(form); };
  int form = chunks > kPiece ? kSmallSlabs : kSmallOne;
  if (!in_one_round(form)) {
    if (D == 128 && in_one_round(kSmallHalfSlabs))
      form = kSmallHalfSlabs;
    else
      form = chunks > kPiece || places(kSmallPairSlabs) > places(kSmallPair) ? kSmallPairSlabs : kSmallPair;
  }
  const size_t lds_bytes = small_lds(D, p.F, chunks, form);
  if (lds_bytes > kMaxLdsBytes) return 1;
  p.units = places(form);
  const int64_t pairs = (p.M + 63) / 64;  // (workgroups take one tile while one round of them suffices)
  const dim3 grid(static_cast<uint32_t>(small_pairs(form) ? std::max<int64_t>(pairs, p.units) : tiles * splits));
#define TAAC_SMALL_LAUNCH(DD, OO, FF, FORM)                                                                           \
  do {                                                                                                                \
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(swiglu_ffn_small_kernel<DD, OO, FF, FORM>),                 \
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)) != hipSuccess)   \
      return set_error(TAAC_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", name, lds_bytes);                      \
    hipLaunchKernelGGL((swiglu_ffn_small_kernel<DD, OO, FF, FORM>), grid, dim3(DD / 32 * kWave), lds_bytes, s, p);    \
    return check_launch(name);                                                                                        \
  } while (0)
#define TAAC_SMALL(DD, OO, FF)                                        \
  do {                                                                \
    if (form == kSmallSlabs) TAAC_SMALL_LAUNCH(DD, OO, FF, kSmallSlabs); \
    if constexpr (DD == 128)                                             \
      if (form == kSmallHalfSlabs) TAAC_SMALL_LAUNCH(DD, OO, FF, kSmallHalfSlabs); \
    if (form == kSmallPair) TAAC_SMALL_LAUNCH(DD, OO, FF, kSmallPair);   \
    if (form == kSmallPairSlabs) TAAC_SMALL_LAUNCH(DD, OO, FF, kSmallPairSlabs);   \
    TAAC_SMALL_LAUNCH(DD, OO, FF, kSmallOne);                         \
  } while (0)
#define TAAC_SMALL_D(DD)                        \
  do {                                          \
    if (with_proj && act_folded) TAAC_SMALL(DD, true, true);   \
    if (with_proj) TAAC_SMALL(DD, true, false);                \
    if (act_folded) TAAC_SMALL(DD, false, true);               \
    TAAC_SMALL(DD, false, false);                              \
  } while (0)
  if (D == 256) TAAC_SMALL_D(256);
  TAAC_SMALL_D(128);
#undef TAAC_SMALL_D
#undef TAAC_SMALL
#undef TAAC_SMALL_LAUNCH
}

}  // namespace taac
