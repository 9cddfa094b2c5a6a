// Fragment-order packing of the token-stationary kernels' weights, one 16-byte piece per call, from bf16 weights or float32
// masters (rounded to bf16 as they are read).
#pragma once

#include "ts_dense.h"

namespace taac {
namespace {

__device__ __forceinline__ bf16x8 weight_piece(const bf16_t* src) { return *reinterpret_cast<const bf16x8*>(src); }
__device__ __forceinline__ bf16x8 weight_piece(const float* src) {
  const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = static_cast<bf16_t>(lo[e]);
    v[4 + e] = static_cast<bf16_t>(hi[e]);
  }
  return v;
}

// ---- fragment-order packing ------------------------------------------------------------------------------------------
// FFN blob: step s (32 hidden units) holds, for chunk q = 0, 1: KS up fragments (k-step r) then MB down fragments
// (row block r - KS); exactly the image one barrier step needs in LDS. A fragment is 64 lanes x 16 bytes.
// col_scale (optional, [D]): weight of the RMSNorm in front of the up projection, folded into its fragments (see
// linear_pack_piece).
// fold_act: the constants of the gate's activation join the same rounding - the gated half is multiplied by -log2(e), the
// other half by -ln 2, so that silu(g) * u = g' * u' / (1 + 2^g') with g' and u' as they leave the matrix unit (the
// kernel's FOLD form: one multiplication less per hidden unit and token; the first-layer bias is scaled when it is staged).
template <typename TW>
__device__ __forceinline__ void ffn_pack_piece(const TW* __restrict__ w_up, const TW* __restrict__ w_down,
                                               bf16x8* __restrict__ packed, int D, int F, int gate_first, int64_t gid,
                                               const TW* __restrict__ col_scale = nullptr, bool fold_act = false) {
  const int KS = D / 16, MB = D / 32, CFRAG = KS + MB, NFRAG = kCPB * CFRAG;
  const int lane = static_cast<int>(gid % 64);
  const int f = static_cast<int>((gid / 64) % NFRAG);
  const int64_t step = gid / 64 / NFRAG;
  const int q = f / CFRAG, r = f % CFRAG;
  const int64_t unit0 = (step * kCPB + q) * kHU;
  const int l32 = lane % 32, hh = lane / 32;
  const TW* src;
  if (r < KS)
    src = w_up + (((l32 < 16) == (gate_first != 0) ? 0 : F) + unit0 + up_unit_of_slot(l32 & 15)) * D + r * 16 + hh * 8;
  else
    src = w_down + static_cast<int64_t>((r - KS) * 32 + l32) * F + unit0 + hh * 8;
  bf16x8 v = weight_piece(src);
  if ((col_scale != nullptr || fold_act) && r < KS) {
    bf16x8 g;
    if (col_scale != nullptr) {
      g = weight_piece(col_scale + r * 16 + hh * 8);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) g[e] = static_cast<bf16_t>(1.0f);
    }
    const float c = fold_act ? (l32 < 16 ? kFoldGate : kFoldValue) : 1.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) * static_cast<float>(g[e]) * c);
  }
  packed[gid] = v;
}

// Linear blob: chunk c (64 output features) holds fragments (row block rb, k-step ks) at index rb * KS + ks.
// col_scale (optional, [K]): every weight is multiplied by the factor of its input feature and rounded once - the weight
// of an RMSNorm in front of the layer, folded into the layer (linear(x * r * g) = r * linear_g(x) with linear_g's weights
// w[n, k] * g[k]; the kernel then applies the per-token factor r to its accumulators).
template <typename TW>
__device__ __forceinline__ void linear_pack_piece(const TW* __restrict__ w, bf16x8* __restrict__ packed, int K, int64_t gid,
                                                  const TW* __restrict__ col_scale = nullptr) {
  const int KS = K / 16, NFRAG = 2 * KS;
  const int lane = static_cast<int>(gid % 64);
  const int f = static_cast<int>((gid / 64) % NFRAG);
  const int64_t chunk = gid / 64 / NFRAG;
  const int l32 = lane % 32, hh = lane / 32;
  const int col = (f % KS) * 16 + hh * 8;
  bf16x8 v = weight_piece(w + (chunk * kNC + (f / KS) * 32 + l32) * K + col);
  if (col_scale != nullptr) {
    const bf16x8 g = weight_piece(col_scale + col);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) * static_cast<float>(g[e]));
  }
  packed[gid] = v;
}

// Feed-forward backward (ffn_bwd.hip). Blob: step s (32 hidden units), sub-step u (k-steps 8 u .. 8 u + 7) holds fragments (block b, k-step 8 u + j) at index
// b * 8 + j; block 0 = rows 32 s .. of the first half of w_up, block 1 = the same rows of its second half, block 2 =
// columns 32 s .. of w_down (rows of its transpose). Lane (l32, hh) of a fragment holds k = 16 ks + 8 hh .. + 7 of row l32.
constexpr int kBwdUnits = 32;   // hidden units per step
constexpr int kBwdSubK = 8;     // k-steps (of 16 features) per sub-step
template <typename TW>
__device__ __forceinline__ void ffn_bwd_pack_piece(const TW* __restrict__ w_up, const TW* __restrict__ w_down,
                                                   bf16x8* __restrict__ packed, int D, int F, int64_t gid) {
  const int NSUB = D / 16 / kBwdSubK, NFRAG = 3 * kBwdSubK;
  const int lane = static_cast<int>(gid % 64);
  const int f = static_cast<int>((gid / 64) % NFRAG);
  const int64_t sub = gid / 64 / NFRAG;  // step * NSUB + u
  const int64_t step = sub / NSUB;
  const int b = f / kBwdSubK, ks = static_cast<int>(sub % NSUB) * kBwdSubK + f % kBwdSubK;
  const int l32 = lane % 32, hh = lane / 32;
  const int64_t unit = step * kBwdUnits + l32;
  const int k0 = ks * 16 + hh * 8;
  bf16x8 v;
  if (b < 2) {
    v = weight_piece(w_up + (b * static_cast<int64_t>(F) + unit) * D + k0);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(w_down[static_cast<int64_t>(k0 + e) * F + unit]);
  }
  packed[gid] = v;
}

}  // namespace
}  // namespace taac
