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
  const int64_t count = token_count(p);
  const int64_t tok0 = static_cast<int64_t>(blockIdx.x) * 32;
  if (tok0 >= count) return;  // whole workgroup
  int64_t xrow[1], prow[4];   // memory rows: of x for token l32; of out / residual for token 8 * i + lane / 8
  TokenRows<1> xr;
  TokenRows<4> pr;
  xr.request(p.x_rows != nullptr ? p.x_rows : p.rows, count, [&](int) { return tok0 + l32; });
  pr.request(p.rows, count, [&](int i) { return tok0 + i * 8 + lane / 8; });
  xr.arrive();
  pr.arrive();
  xrow[0] = xr.row(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) prow[i] = pr.row(i);
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
        if (hh == 0) p.qk_sumsq[static_cast<int64_t>(chunk) * p.M + row] = ss;
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

}  // namespace

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

}  // namespace taac
