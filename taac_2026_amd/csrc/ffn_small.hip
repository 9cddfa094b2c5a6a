// Dense kernels of the token path for few tokens (gfx950, model width D = 256 or 128).
//
// The kernels of ffn.hip keep 256 or 512 tokens in a workgroup and stream the weights past them: the right shape when every
// compute unit has a tile, and a long serial walk over the weights by a handful of compute units when a batch holds a
// few thousand tokens or one request. Here the work of a 32-token tile is spread instead: the wavefronts of a workgroup share
// the tokens and divide the OUTPUT features (projection), so that each reads its own slice of the packed weights
// straight from L2 into MFMA operand registers - fragments are 1 KB of contiguous memory, no other wavefront of the workgroup
// wants them, so a stop in LDS would only add a barrier. What bounds these kernels is latency: row count -> row index ->
// token rows -> products -> store, with the weight fragments requested in front of that chain.
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

// [RMSNorm (weight folded) ->] linear [-> + residual], K = D, weights in fragment order. A workgroup takes 32 tokens
// (blockIdx.x) and D output features (blockIdx.y), 64 per wavefront. QK as in norm_linear_kernel: the features of the query
// (blockIdx.y = 0) and of the key (1) leave their sum of squares behind - as the norm's factor per token in qk_rstd when that
// is given (the workgroup holds all features of the part), per 64-feature chunk in qk_sumsq otherwise - and with QK == 2 are
// multiplied by the norm weight and rotated. Same values as norm_linear_kernel, bit for bit (same products in the same order).
// q | k | v of one request (512 tokens, D = 256): 6.0 us, the persistent kernel 13.6; its line is at dense_few_rows.
template <int D, bool RES, int QK>
__global__ __launch_bounds__(D, 2) void norm_linear_small_kernel(const TsParams p) {
  constexpr int NW = D / kNC;  // wavefronts
  constexpr int KS = D / 16;
  constexpr int NFRAG = 2 * KS;
  __shared__ __attribute__((aligned(16))) uint8_t tiles[NW * kStageWave];
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

  // The weights depend on nothing: requested first, in flight behind the row count and the row index.
  const char* wsrc = reinterpret_cast<const char*>(p.w1) + static_cast<int64_t>(chunk) * NFRAG * kFrag;
  bf16x8 w[NFRAG];
#pragma unroll
  for (int i = 0; i < NFRAG; ++i) w[i] = *reinterpret_cast<const bf16x8*>(wsrc + i * kFrag + lane * 16);
  __builtin_amdgcn_sched_barrier(0);
  const int64_t tok0 = static_cast<int64_t>(blockIdx.x) * 32;
  SmallRows<1> xr;  // memory rows: of x for token l32; of out / residual for token 8 * i + lane / 8
  SmallRows<4> pr;
  xr.request(p, p.x_rows != nullptr ? p.x_rows : p.rows, [&](int) { return tok0 + l32; });
  pr.request(p, p.rows, [&](int i) { return tok0 + i * 8 + lane / 8; });
  const int64_t count = token_count(p);
  if (tok0 >= count) return;  // whole workgroup
  int64_t xrow[1], prow[4];
  xr.resolve(count, xrow);
  pr.resolve(count, prow);
  bf16x8 xf[1][KS];
  load_token_rows_at<D, 1>(p, xrow, hh, xf);
  const bf16_t* bias = p.b1 != nullptr ? p.b1 + chunk * kNC : nullptr;
  bf16x4 bv[8];
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) bv[q][e] = static_cast<bf16_t>(0.f);
  if (bias != nullptr) read_chunk_bias(bias, hh, bv);
  bf16x8 res[4];
  if constexpr (RES) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      res[i] = *reinterpret_cast<const bf16x8*>(p.residual + prow[i] * p.ldr + chunk * kNC + (lane % 8) * 8);
  }

  f32x16 acc0, acc1;
#pragma unroll
  for (int j = 0; j < 16; ++j) acc0[j] = acc1[j] = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ks], xf[0][ks], acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[KS + ks], xf[0][ks], acc1, 0, 0, 0);
  }
  float rstd[1] = {1.0f};
  if (p.norm_w != nullptr) token_rstd<D, 1>(p.eps, xf, rstd);  // the norm's weight is part of the packed layer
  if (p.rstd_out != nullptr && part == 0 && wave == 0 && hh == 0 && tok0 + l32 < count)
    p.rstd_out[token_row(p, count, tok0 + l32)] = rstd[0];

  uint8_t* tile = tiles + wave * kStageWave;
  [[maybe_unused]] const bool qk_part = QK != 0 && chunk < p.qk_chunks;  // the same for all wavefronts of a part
  if constexpr (QK != 0) {
    if (qk_part && (p.qk_sumsq != nullptr || p.qk_rstd != nullptr)) {
      const float ss = half_wave_pair_sum(tile_to_lds_sumsq(tile, acc0, acc1, bv, l32, hh, rstd[0]));
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
      tile_to_lds(tile, acc0, acc1, bv, l32, hh, rstd[0]);
    }
  } else {
    tile_to_lds(tile, acc0, acc1, bv, l32, hh, rstd[0]);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (!active) return;  // no barrier below
  const int col8 = chunk * kNC + (lane % 8) * 8;
  [[maybe_unused]] bf16x8 wn;
  [[maybe_unused]] bool rotate = false;
  if constexpr (QK == 2) {
#pragma unroll
    for (int e = 0; e < 8; ++e) wn[e] = static_cast<bf16_t>(1.0f);
    if (qk_part && p.qk_w != nullptr)
      wn = *reinterpret_cast<const bf16x8*>(part == 0 ? p.qk_w + col8 : p.qk_wk + (col8 - D));
    rotate = qk_part && p.cos_sin != nullptr;
  }
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
          const bf16x8 cs = *reinterpret_cast<const bf16x8*>(p.cos_sin + static_cast<int64_t>(pos) * p.head_dim + col8 % p.head_dim);
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
    // feature planes: column col8 lies in plane col8 >> shift, at col8 % 2^shift of the row
    const int64_t at = p.out_plane_shift > 0
                           ? (((static_cast<int64_t>(col8 >> p.out_plane_shift) * p.M + prow[i]) << p.out_plane_shift) +
                              (col8 & ((1 << p.out_plane_shift) - 1)))
                           : prow[i] * p.ldo + col8;
    *reinterpret_cast<bf16x8*>(p.out + at) = v;
  }
}

// Data that other workgroups of the same launch read: accesses at the scope of the whole chip, which go through the L2 of the die
// to the memory all dies share. (Ordinary stores with a fence behind them write back and drop everything the die's L2 holds:
// 8 us per launch.)
// Sixteen bytes per lane and access: as atomic accesses, eight bytes at most, twice as many requests leave the compute unit and the
// last workgroup of a tile takes 5 us for its 256 KB (512 tokens, D = 256, F = 1024, eight splits: 19.7 -> 17.0 us for the kernel).
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
// 32 tokens per workgroup (the products, blobs and roundings of swiglu_ffn_kernel). Four wavefronts share the tokens and divide
// the HIDDEN units: wavefront w takes the 16-unit chunks w, w + 4, ...; each holds a [D, 32] partial of the down projection
// in its accumulators, and the four partials meet once, in LDS, where every wavefront adds up its share of the features in a
// fixed order. The projection in front is divided by output features; its result reaches the other wavefronts through LDS.
// A wavefront is alone on its SIMD and reads its fragments from L2 through a ring as deep as a chunk (24 KB in flight at
// D = 256, 96 KB per compute unit).
// Bound: the 1.6 MB of weights a compute unit pulls from L2 for its 32 tokens (0.7 us per chunk and wavefront, 64 bytes per
// clock of the compute unit: 11 us) behind and in front of which lie 9.5 us of latency chains; the persistent kernel has one
// or two of its eight wavefronts at work there and takes 50 us whatever the number of tokens (512 tokens, D = 256, F = 1024:
// 49.9 -> 21.5 us; 8192 tokens: 55.6 -> 27.8; its line is at ffn_few_rows).
// splits > 1 (see TsParams): for batches that leave most of the chip idle even so, the hidden units of a tile are also divided over
// workgroups, eight at most (one request of 512 positions, eight splits, with the requests below ordered by need: the whole
// 4-block call 164 -> 140 us; fences instead of the write-through accesses: 156; those accesses 16 bytes wide instead
// of 8: 128 -> 119). Sixteen lose where tiles and F admit them: a wavefront then has one 16-unit chunk behind the same latency
// chains (with 8-byte accesses, F = 1024 160 against 140 us for eight, F = 2048 169 against 151). At F = 512 eight leave it one chunk, too,
// and cost 4 % (at most 8 / 4 / 2 splits, one request of 512 positions, D = 256: F = 512 137 / 132 / 134 us, F = 1024 142 / 141 / 150,
// F = 2048 156 / 161 / 183; D = 128: F = 512 99 / 96 / 95, F = 1024 102 / 100 / 104); another number would add the units in another
// order and move every output by roundings.
// LDS: [4 partials of 32 x D floats][x1 (32 padded rows of D bf16)][first-layer bias 2F][4 x 32 row sums]
// ------------------------------------------------------------------------------------------------------------------
template <int D, bool OUTP, bool FOLD>
__global__ __launch_bounds__(4 * kWave, 1) void swiglu_ffn_small_kernel(const TsParams p) {
  constexpr int NW = 4;
  constexpr int KS = D / 16, MB = D / 32;
  constexpr int CFRAG = KS + MB;
  constexpr int MBW = MB / NW;              // 32-feature blocks a wavefront projects in front and adds up behind
  constexpr int kRow = D * 2 + 16;          // bytes per row of the x1 tile
  constexpr int kPart = MB * 4 * kWave * 16;  // bytes of one partial
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  uint8_t* x1_lds = smem + NW * kPart;
  bf16_t* bias_lds = reinterpret_cast<bf16_t*>(x1_lds + 32 * kRow);
  float* sums = reinterpret_cast<float*>(bias_lds + 2 * p.F);  // [NW][32]

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int l32 = lane % 32, hh = lane / 32;
  const int F = p.F;
  const int nchunks = F / kHU;

  // Requests in the order in which their values are needed (they arrive in that order): row index and count, the projection's
  // weights behind them, then - one latency later - the token rows, and last what is used after the projection.
  const int64_t tok0 = static_cast<int64_t>(blockIdx.x) * 32;
  SmallRows<1> xr, orow;
  xr.request(p, p.x_rows != nullptr ? p.x_rows : p.rows, [&](int) { return tok0 + l32; });
  orow.request(p, p.rows, [&](int) { return tok0 + l32; });
  const int64_t count = token_count(p);
  __builtin_amdgcn_sched_barrier(0);
  [[maybe_unused]] bf16x8 w0[OUTP ? MBW * KS : 1];
  if constexpr (OUTP) {
    const char* src = reinterpret_cast<const char*>(p.w0) + static_cast<int64_t>(wave * MBW * KS) * kFrag;
#pragma unroll
    for (int i = 0; i < MBW * KS; ++i) w0[i] = *reinterpret_cast<const bf16x8*>(src + i * kFrag + lane * 16);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (tok0 >= count) return;  // whole workgroup
  int64_t xrow[1], orows[1];
  xr.resolve(count, xrow);
  orow.resolve(count, orows);
  const int64_t row = orows[0];  // of token l32 in residual / out
  bf16x8 xf[1][KS];
  load_token_rows_at<D, 1>(p, xrow, hh, xf);
  // Four features per register quad of the lane's blocks, in accumulator order. A vector that is absent is read from the weights
  // instead (finite, in bounds for D values) and cleared where it is used: no branch between the loads.
  auto feature_vectors = [&](const bf16_t* v, bf16x4 (&dst)[MBW][4]) {
    const bf16_t* src = v != nullptr ? v : p.w1;
#pragma unroll
    for (int m = 0; m < MBW; ++m)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq)
        dst[m][jq] = *reinterpret_cast<const bf16x4*>(src + (wave * MBW + m) * 32 + jq * 8 + hh * 4);
  };
  [[maybe_unused]] bf16x4 hv[MBW][4], b0v[MBW][4];  // block input, projection bias
  if constexpr (OUTP) {
    feature_vectors(p.residual + row * p.ldr, hv);
    feature_vectors(p.b0, b0v);
  }
  __builtin_amdgcn_sched_barrier(0);
  const int splits = p.splits > 1 ? p.splits : 1;
  const int first_chunk = static_cast<int>(blockIdx.y) * NW + wave, stride = NW * splits;
  const int first = first_chunk < nchunks ? first_chunk : nchunks - 1;
  const char* ffn_blob = reinterpret_cast<const char*>(p.w1) + lane * 16;
  bf16x8 ring[CFRAG];
  auto load_chunk_frag = [&](int chunk, int i) {
    return *reinterpret_cast<const bf16x8*>(ffn_blob + (static_cast<int64_t>(chunk) * CFRAG + i) * kFrag);
  };
#pragma unroll
  for (int i = 0; i < CFRAG; ++i) ring[i] = load_chunk_frag(first, i);
  // first-layer bias, gated half first; FOLD: with the constants the packed layer carries. 8 entries per thread and round.
  auto bias_piece = [&](int i) {
    const bool gated = i < F;  // F is a multiple of 32: a piece lies in one half
    return *reinterpret_cast<const bf16x8*>(p.b1 != nullptr ? p.b1 + (gated == (p.gate_first != 0) ? i % F : F + i % F) : p.w1);
  };
  auto store_bias = [&](int i, bf16x8 v) {
    const float c = p.b1 == nullptr ? 0.f : (!FOLD ? 1.f : (i < F ? kFoldGate : kFoldValue));
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) * c);
    if (i < 2 * F) *reinterpret_cast<bf16x8*>(bias_lds + i) = v;
  };
  const bf16x8 bias_regs = bias_piece(tid * 8 < 2 * F ? tid * 8 : 0);
  bf16x4 b2v[MBW][4], hwv[MBW][4];  // for the end of the kernel: down-projection bias, readout weight
  feature_vectors(p.b2, b2v);
  feature_vectors(p.head_w, hwv);
  __builtin_amdgcn_sched_barrier(0);

  if constexpr (OUTP) {
    const float b0_on = p.b0 != nullptr ? 1.f : 0.f;
    float ss = 0.f;
#pragma unroll
    for (int m = 0; m < MBW; ++m) {
      f32x16 acc;
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0[m * KS + ks], xf[0][ks], acc, 0, 0, 0);
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        bf16x4 x1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lin = static_cast<float>(static_cast<bf16_t>(fmaf(static_cast<float>(b0v[m][jq][e]), b0_on, acc[jq * 4 + e])));
          x1[e] = static_cast<bf16_t>(lin + static_cast<float>(hv[m][jq][e]));
          const float r = static_cast<float>(x1[e]);
          ss = fmaf(r, r, ss);
        }
        *reinterpret_cast<bf16x4*>(x1_lds + l32 * kRow + ((wave * MBW + m) * 32 + jq * 8 + hh * 4) * 2) = x1;
      }
    }
    ss = half_wave_pair_sum(ss);
    if (hh == 0) sums[wave * 32 + l32] = ss;
  }
  store_bias(tid * 8, bias_regs);
  for (int i = (NW * kWave + tid) * 8; i < 2 * F; i += NW * kWave * 8) store_bias(i, bias_piece(i));
  __syncthreads();
  if constexpr (OUTP) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) total += sums[w * 32 + l32];
    const float scale = p.norm_w != nullptr ? rsqrtf(total * (1.0f / D) + p.eps) : 1.0f;
    if (p.rstd_out != nullptr && wave == 0 && hh == 0 && tok0 + l32 < count) p.rstd_out[row] = scale;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      xf[0][ks] = *reinterpret_cast<const bf16x8*>(x1_lds + l32 * kRow + (ks * 16 + hh * 8) * 2);
#pragma unroll
      for (int e = 0; e < 8; ++e) xf[0][ks][e] = static_cast<bf16_t>(static_cast<float>(xf[0][ks][e]) * scale);
    }
  } else if (p.norm_w != nullptr) {
    float rstd[1];
    token_rstd<D, 1>(p.eps, xf, rstd);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) xf[0][ks][e] = static_cast<bf16_t>(static_cast<float>(xf[0][ks][e]) * rstd[0]);
  }

  f32x16 oacc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < 16; ++j) oacc[mb][j] = 0.f;
  for (int chunk = first_chunk; chunk < nchunks; chunk += stride) {
    const int next = chunk + stride < nchunks ? chunk + stride : chunk;  // the last chunk is requested once more, and not used
    const bf16x8 bg = *reinterpret_cast<const bf16x8*>(bias_lds + chunk * kHU + hh * 8);
    const bf16x8 bu = *reinterpret_cast<const bf16x8*>(bias_lds + F + chunk * kHU + hh * 8);
    f32x16 gu;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      gu[e] = static_cast<float>(bg[e]);
      gu[8 + e] = static_cast<float>(bu[e]);
    }
    static_for<KS>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      gu = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i], xf[0][i], gu, 0, 0, 0);
      ring[i] = load_chunk_frag(next, i);
      __builtin_amdgcn_sched_barrier(0);
    });
    bf16x8 hb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (FOLD)
        hb[e] = static_cast<bf16_t>(gu[e] * gu[8 + e] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gu[e])));
      else
        hb[e] = static_cast<bf16_t>(silu_f(gu[e]) * gu[8 + e]);
    }
    static_for<MB>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      oacc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[KS + i], hb, oacc[i], 0, 0, 0);
      ring[KS + i] = load_chunk_frag(next, KS + i);
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // ---- the four partials: [wavefront][feature block][register quad][lane] -------------------------------------------------
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const f32x4 v = {oacc[mb][jq * 4], oacc[mb][jq * 4 + 1], oacc[mb][jq * 4 + 2], oacc[mb][jq * 4 + 3]};
      *reinterpret_cast<f32x4*>(smem + wave * kPart + ((mb * 4 + jq) * kWave + lane) * 16) = v;
    }
  __syncthreads();
  f32x4 total[MBW][4];
#pragma unroll
  for (int m = 0; m < MBW; ++m)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const int piece = ((wave * MBW + m) * 4 + jq) * kWave + lane;
      total[m][jq] = *reinterpret_cast<const f32x4*>(smem + piece * 16);
#pragma unroll
      for (int w = 1; w < NW; ++w) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(smem + w * kPart + piece * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) total[m][jq][e] += v[e];
      }
    }
  if (splits > 1) {
    // The partial of this workgroup becomes visible to the chip, then the workgroup counts itself: whoever counts last finds all
    // partials of the tile (nobody waits for anybody). They are added in the order of the splits: the same result every run.
    const SharedPartials parts(p.split_partials + static_cast<int64_t>(blockIdx.x) * splits * (kPart / 4), splits * kPart);
    const int lane_at = (wave * MBW * 4 * kWave + lane) * 16;  // of a partial: [feature block][register quad][lane]
    const int mine = static_cast<int>(blockIdx.y) * kPart + lane_at;
#pragma unroll
    for (int m = 0; m < MBW; ++m)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) parts.store(mine + (m * 4 + jq) * (kWave * 16), total[m][jq]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's partials have reached the chip's common memory
    __syncthreads();
    uint32_t* arrived = reinterpret_cast<uint32_t*>(sums);
    if (tid == 0)
      *arrived = __hip_atomic_fetch_add(p.split_counters + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const bool last = *arrived == static_cast<uint32_t>(splits - 1);
    __syncthreads();  // (the row sums of the readout reuse the word)
    if (!last) return;
    if (tid == 0) p.split_counters[blockIdx.x] = 0u;
#pragma unroll
    for (int m = 0; m < MBW; ++m)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq)
#pragma unroll
        for (int e = 0; e < 4; ++e) total[m][jq][e] = 0.f;
    auto add_partials = [&](int first_split, auto ahead) {
      constexpr int kAhead = decltype(ahead)::value;  // partials in flight
      f32x4 v[kAhead][MBW][4];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
#pragma unroll
        for (int m = 0; m < MBW; ++m)
#pragma unroll
          for (int jq = 0; jq < 4; ++jq)
            v[u][m][jq] = parts.load((first_split + u) * kPart + lane_at + (m * 4 + jq) * (kWave * 16));
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
#pragma unroll
        for (int m = 0; m < MBW; ++m)
#pragma unroll
          for (int jq = 0; jq < 4; ++jq)
#pragma unroll
            for (int e = 0; e < 4; ++e) total[m][jq][e] += v[u][m][jq][e];
    };
    // 2, 4 or 8 splits (ffn_splits). Eight partials, 64 KB per wavefront: 17.0 us for the kernel with four in flight, 17.5 with two.
    if (splits == 2) add_partials(0, std::integral_constant<int, 2>{});
    for (int w = 0; w + 4 <= splits; w += 4) add_partials(w, std::integral_constant<int, 4>{});
  }
  const bool live = tok0 + l32 < count;
  if (OUTP && p.x1_out != nullptr) {
    for (int idx = tid; idx < 32 * (D / 8); idx += NW * kWave) {
      const int t = idx / (D / 8), c = idx % (D / 8) * 8;
      if (tok0 + t >= count) continue;
      const int64_t r = p.rows != nullptr ? static_cast<int64_t>(p.rows[tok0 + t]) : tok0 + t;
      *reinterpret_cast<bf16x8*>(p.x1_out + r * D + c) = *reinterpret_cast<const bf16x8*>(x1_lds + t * kRow + c * 2);
    }
  }
  const float b2_on = p.b2 != nullptr ? 1.f : 0.f;
  float hdot = 0.f;
#pragma unroll
  for (int m = 0; m < MBW; ++m)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const int col = (wave * MBW + m) * 32 + jq * 8 + hh * 4;
      f32x4 s = total[m][jq];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = fmaf(static_cast<float>(b2v[m][jq][e]), b2_on, s[e]);
      bf16x4 o;
      if constexpr (OUTP) {  // x1 + down, rounded once
        const bf16x4 x1 = *reinterpret_cast<const bf16x4*>(x1_lds + l32 * kRow + col * 2);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16_t>(s[e] + static_cast<float>(x1[e]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16_t>(s[e]);
        if (p.residual != nullptr) {
          const bf16x4 r = *reinterpret_cast<const bf16x4*>(p.residual + row * p.ldr + col);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16_t>(static_cast<float>(o[e]) + static_cast<float>(r[e]));
        }
      }
      if (live) *reinterpret_cast<bf16x4*>(p.out + row * p.ldo + col) = o;
#pragma unroll
      for (int e = 0; e < 4; ++e) hdot = fmaf(static_cast<float>(o[e]), static_cast<float>(hwv[m][jq][e]), hdot);
    }
  if (p.head_w != nullptr) {
    hdot = half_wave_pair_sum(hdot);
    if (hh == 0) sums[wave * 32 + l32] = hdot;
    __syncthreads();
    if (wave == 0 && hh == 0 && live) {
      float d = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) d += sums[w * 32 + l32];
      p.token_dots[row] = d;
    }
  }
}

}  // namespace

int ffn_splits(int64_t M, int32_t D, int32_t F) {
  const int64_t tiles = (M + 31) / 32;
  const int cus = compute_units();
  int splits = 1;
  if (ffn_few_rows(M, D))
    while (splits < 8 && 2 * splits * tiles <= cus && 2 * splits * 4 * kHU <= F) splits *= 2;
  return splits;
}

int64_t ffn_split_bytes(int64_t M, int32_t D, int32_t F) {
  const int splits = ffn_splits(M, D, F);
  if (splits == 1) return 0;
  const int64_t tiles = (M + 31) / 32;
  return tiles * splits * 32 * D * 4 + (tiles * 4 + 255) / 256 * 256;
}

int norm_linear_small(const TsParams& p, int32_t K, int qk_mode, hipStream_t s, const char* name) {
  const dim3 grid(static_cast<uint32_t>((p.M + 31) / 32), static_cast<uint32_t>((p.N + K - 1) / K));
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

int swiglu_ffn_small(const TsParams& p, int32_t D, bool with_proj, bool act_folded, hipStream_t s, const char* name) {
  const size_t lds_bytes = static_cast<size_t>(4) * 32 * D * 4 + 32 * (D * 2 + 16) + static_cast<size_t>(2) * p.F * 2 + 4 * 32 * 4;
  if (lds_bytes > 160 * 1024) return 1;
  const dim3 grid(static_cast<uint32_t>((p.M + 31) / 32), p.splits > 1 ? p.splits : 1);
#define TAAC_SMALL(DD, OO, FF)                                                                                        \
  do {                                                                                                                \
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(swiglu_ffn_small_kernel<DD, OO, FF>),                       \
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)) != hipSuccess)   \
      return set_error(TAAC_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", name, lds_bytes);                      \
    hipLaunchKernelGGL((swiglu_ffn_small_kernel<DD, OO, FF>), grid, dim3(4 * kWave), lds_bytes, s, p);                \
    return check_launch(name);                                                                                        \
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
}

}  // namespace taac
