// Dense backward kernels of the training stack (see train_ops.h): the input gradient of a normalised layer with the norm's
// backward and the residual gradient in its epilogue, and the weight gradients of a block's four layers in one launch.
#include "train_ops.h"
#include "ts_common.h"

namespace taac {
namespace {

// ------------------------------------------------------------------------------------------------------------------
// dx = dres + rstd * (g - x_hat * mean(g * x_hat)),  g = (dy W) * norm_w,  x_hat = x * rstd.
//
// The product is the narrow output of a long contraction (K = 2F or 3D, D features): a workgroup takes 64 * TG tokens x all
// features, so dy is read once and complete rows meet in the workgroup; TG token groups of 64 x FG feature groups, a wavefront
// each. K is walked in slabs: both operands' slabs go from global memory straight into LDS (1 KB per transfer) into a ring of
// stages, RING - 1 slabs ahead; the 16-byte pieces of a row are XOR-swizzled by its number, so that the 16 lanes of a fragment
// read hit distinct banks. Rows beyond the count repeat the last row and are not stored.
// The epilogue replaces a store of dh = dy W, the norm's backward over x and dh, and the residual add: 3 of the 8 passes over
// [M, D] that the layer-by-layer backward makes here. The gradient of the norm's weight is left to the weight-gradient kernels,
// which hold sum_m dy[m, n] x_hat[m, k] anyway (d norm_w[k] = sum_n w[n, k] of it).
// The epilogue's rows pass through LDS: read and written as a lane's own eight bytes of 32 rows at once, they cost 46 us per
// 256-token workgroup whatever K (294 912 tokens, D = 256: K = 768 337 -> 220 us, K = 2048 515 -> 400 us).
// Bound: HBM (dy, K * 2 bytes per token). Where 256-token workgroups would leave compute units idle a workgroup takes 64 tokens,
// and a slab's chain (barrier, fragment reads, products, transfers) is the time: eight wavefronts and slabs of 64 columns instead
// of two and 32, 6 100 tokens, D = 256: K = 2048 43 -> 24 us.
// The weight lies in panels of 32 columns (transposed_weight_at): a slab of it is one or two runs of memory. As rows of K columns its
// D pieces of 64 or 128 bytes were a power of two apart and came from the same memory channels: 285 000 tokens, D = 256: K = 2048
// 401 -> 379 us, K = 768 207 -> 197; 30 000 tokens, both 42.6 -> 38.5.
// ------------------------------------------------------------------------------------------------------------------

struct DgradParams {
  const bf16_t* dy;
  const bf16_t* w_t;
  const bf16_t* x;
  const float* rstd;
  const bf16_t* norm_w;
  const bf16_t* dres;
  bf16_t* dx;
  const int32_t* count;
  int64_t M;
  int32_t K;
  bool panels;           // dy in panel order
};

// TG: token groups of 64; FG: feature groups (wavefronts = TG * FG); SLAB: columns of dy per stage, RING stages.
template <int D, int TG, int FG, int SLAB, int RING>
__global__ __launch_bounds__(TG * FG * kWave, 2) void dgrad_norm_kernel(const DgradParams p) {
  constexpr int NWAVES = TG * FG;
  constexpr int TOK = 64 * TG;
  constexpr int NI = D / FG / 32;               // 32-feature blocks per wavefront
  constexpr int kRowB = SLAB * 2;               // bytes of a staged row
  constexpr int kTokBytes = TOK * kRowB, kStage = kTokBytes + D * kRowB;
  constexpr int LPR = SLAB / 8, RPX = kWave / LPR;  // lanes per row and rows per transfer
  constexpr int AT = TOK / RPX / NWAVES, WT = D / RPX / NWAVES;  // transfers per wavefront and slab: rows of dy, of the weight
  constexpr int PW = AT + WT;
  static_assert(TOK % (RPX * NWAVES) == 0 && D % (RPX * NWAVES) == 0, "every wavefront stages the same number of pieces");
  static_assert((SLAB == 32 || SLAB == 64) && SLAB % kPanelCols == 0 && kPanelRows % TOK == 0, "a slab of a workgroup lies in whole panel rows");
  static_assert(RING == 3 || RING == 4, "waits are written for these");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

  int64_t rows = p.M;
  {
    const int64_t n = *p.count;
    rows = n < rows ? n : rows;
  }
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * TOK;
  if (m0 >= rows) return;  // whole workgroup
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int l32 = lane % 32, hh = lane / 32;
  const int wt = wave % TG, wn = wave / TG;
  const int nslabs = p.K / SLAB;

  // piece order of a staged row: the 16 rows that a fragment read touches together fall on distinct banks
  auto swizzle = [](int row) { return SLAB == 32 ? (row >> 2) & 3 : (row >> 1) & 7; };
  const bf16_t* a_src[AT];
  const bf16_t* w_src[WT];
#pragma unroll
  for (int i = 0; i < AT; ++i) {
    const int row = RPX * (AT * wave + i) + lane / LPR, piece = (lane % LPR) ^ swizzle(row);
    const int64_t arow = m0 + row < rows ? m0 + row : rows - 1;
    a_src[i] = p.dy + (p.panels ? panel_row(arow, p.K) + piece / 4 * kPanel + piece % 4 * 8 : arow * p.K + piece * 8);
  }
#pragma unroll
  for (int i = 0; i < WT; ++i) {
    const int row = RPX * (WT * wave + i) + lane / LPR;
    w_src[i] = p.w_t + transposed_weight_at(row, ((lane % LPR) ^ swizzle(row)) * 8, D);
  }
  // every workgroup starts its walk over K at a different slab, so that they do not all ask the same memory channels at once
  const int rot = static_cast<int>((blockIdx.x * 5u) % static_cast<uint32_t>(nslabs));
  const int64_t slab_stride = p.panels ? SLAB / kPanelCols * kPanel : SLAB;
  auto stage = [&](int slab) {
    uint8_t* base = smem + (slab % RING) * kStage;
    const int turned = slab + rot;
    const int at = turned >= nslabs ? turned - nslabs : turned;
    const int64_t a0 = at * slab_stride;
    const int64_t w0 = transposed_weight_at(0, static_cast<int64_t>(at) * SLAB, D);
#pragma unroll
    for (int i = 0; i < AT; ++i) lds_dma16(a_src[i] + a0, base + (AT * wave + i) * 1024);
#pragma unroll
    for (int i = 0; i < WT; ++i) lds_dma16(w_src[i] + w0, base + kTokBytes + (WT * wave + i) * 1024);
  };
  const int swz = swizzle(l32);  // of any row l32 + a multiple of 32
  int piece_off[SLAB / 16];
#pragma unroll
  for (int ks = 0; ks < SLAB / 16; ++ks) piece_off[ks] = ((2 * ks + hh) ^ swz) * 16;
  const int a_row_off = (wt * 64 + l32) * kRowB;
  const int w_row_off = kTokBytes + (wn * (D / FG) + l32) * kRowB;

  f32x16 acc[NI][2];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[ni][mi][j] = 0.f;

#pragma unroll
  for (int q = 0; q < RING - 1; ++q)
    if (q < nslabs) stage(q);
  if (RING == 4 && nslabs > 2) vm_wait<2 * PW>();
  else if (nslabs > 1) vm_wait<PW>();
  else vm_wait<0>();
  __syncthreads();
  for (int s = 0; s < nslabs; ++s) {
    if (s + RING - 1 < nslabs) stage(s + RING - 1);  // the slot last read in slab s - 1, which every wavefront has left
    const uint8_t* st = smem + (s % RING) * kStage;
#pragma unroll
    for (int ks = 0; ks < SLAB / 16; ++ks) {
      bf16x8 wf[NI], af[2];
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) af[mi] = *reinterpret_cast<const bf16x8*>(st + a_row_off + mi * 32 * kRowB + piece_off[ks]);
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) wf[ni] = *reinterpret_cast<const bf16x8*>(st + w_row_off + ni * 32 * kRowB + piece_off[ks]);
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) acc[ni][mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ni], af[mi], acc[ni][mi], 0, 0, 0);
    }
    if (s + 1 < nslabs) {
      // the transfers of slab s + 1 were issued RING - 1 slabs ago; behind them are those of slab s + 2 (and s + 3)
      if (RING == 4 && s + 3 < nslabs) vm_wait<2 * PW>();
      else if (s + 2 < nslabs) vm_wait<PW>();
      else vm_wait<0>();
    }
    __syncthreads();
  }

  // acc[ni][mi][jq * 4 + e]: feature wn * D / FG + ni * 32 + jq * 8 + hh * 4 + e of token wt * 64 + mi * 32 + l32.
  // A lane holds eight bytes out of each 32 features of one row, so x, dres and dx pass through LDS, 32 * TG tokens (one mi) at a
  // time over the ring's memory: whole rows in and out of memory, the 16-byte pieces of a tile row XOR-swizzled by row % 16.
  constexpr int TILE_ROWS = 32 * TG, kRowBytes = D * 2, kTile = TILE_ROWS * kRowBytes;
  constexpr int RPT = 1024 / kRowBytes;           // rows per transfer
  constexpr int NT = TILE_ROWS / NWAVES / RPT;    // transfers per wavefront and tile
  constexpr int PIECES = D / 8;
  uint8_t* x_tile = smem;
  uint8_t* res_tile = smem + kTile;
  float* red = reinterpret_cast<float*>(smem + 2 * kTile);  // [FG][TILE_ROWS] sums of g * x
  const int trow = wt * 32 + l32;
  auto token_of = [&](int tile_row, int mi) { return m0 + tile_row / 32 * 64 + mi * 32 + tile_row % 32; };
  auto lane_piece = [&](int ni, int jq) { return trow * kRowBytes + (((wn * (D / FG / 8) + ni * 4 + jq) ^ (trow & 15)) * 16) + hh * 8; };
#pragma unroll
  for (int mi = 0; mi < 2; ++mi) {
    if (mi > 0) __syncthreads();  // the tiles have been stored
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tr = (wave * NT + i) * RPT + lane / PIECES;
      const int64_t m = token_of(tr, mi);
      const int64_t at = (m < rows ? m : rows - 1) * D + ((lane % PIECES) ^ (tr & 15)) * 8;
      lds_dma16(p.x + at, x_tile + (wave * NT + i) * 1024);
      lds_dma16(p.dres + at, res_tile + (wave * NT + i) * 1024);
    }
    const int64_t m = token_of(trow, mi);
    const float scale = p.rstd[m < rows ? m : rows - 1];
    vm_wait<0>();
    __syncthreads();
    float part = 0.f;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        const bf16x4 xv = *reinterpret_cast<const bf16x4*>(x_tile + lane_piece(ni, jq));
        const bf16x4 wv = *reinterpret_cast<const bf16x4*>(p.norm_w + wn * (D / FG) + ni * 32 + jq * 8 + hh * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = acc[ni][mi][jq * 4 + e] * static_cast<float>(wv[e]);
          acc[ni][mi][jq * 4 + e] = g;
          part = fmaf(g, static_cast<float>(xv[e]), part);  // times rstd: x_hat
        }
      }
    const uint32_t u = __builtin_bit_cast(uint32_t, part);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const float both = __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) + __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
    if (hh == 0) red[wn * TILE_ROWS + trow] = both;
    __syncthreads();
    // mean(g * x_hat) * x_hat = (sum of g * x) / D * rstd^2 * x
    float sum = red[trow];
#pragma unroll
    for (int f = 1; f < FG; ++f) sum += red[f * TILE_ROWS + trow];
    const float proj = sum * (1.0f / D) * scale * scale;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        bf16x4* xp = reinterpret_cast<bf16x4*>(x_tile + lane_piece(ni, jq));
        const bf16x4 xv = *xp;
        const bf16x4 rv = *reinterpret_cast<const bf16x4*>(res_tile + lane_piece(ni, jq));
        bf16x4 ov;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          ov[e] = static_cast<bf16_t>(static_cast<float>(rv[e]) +
                                      scale * (acc[ni][mi][jq * 4 + e] - static_cast<float>(xv[e]) * proj));
        *xp = ov;
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tr = (wave * NT + i) * RPT + lane / PIECES;
      const int64_t mo = token_of(tr, mi);
      const bf16x8 ov = *reinterpret_cast<const bf16x8*>(x_tile + tr * kRowBytes + ((lane % PIECES) ^ (tr & 15)) * 16);
      if (mo < rows) *reinterpret_cast<bf16x8*>(p.dx + mo * D + lane % PIECES * 8) = ov;
    }
  }
}

template <int D, int TG, int FG, int SLAB, int RING>
int launch_dgrad(const DgradParams& p, hipStream_t s, const char* name) {
  constexpr size_t ring = static_cast<size_t>(RING) * (64 * TG + D) * SLAB * 2;
  constexpr size_t tiles = static_cast<size_t>(32 * TG) * (2 * D * 2 + FG * sizeof(float));
  constexpr size_t lds = ring > tiles ? ring : tiles;
  auto kernel = dgrad_norm_kernel<D, TG, FG, SLAB, RING>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) !=
      hipSuccess)
    return set_error(TAAC_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", name, lds);
  const int64_t grid = (p.M + 64 * TG - 1) / (64 * TG);
  if (grid > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: too many workgroups", name);
  hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(grid)), dim3(TG * FG * kWave), lds, s, p);
  return check_launch(name);
}

// ------------------------------------------------------------------------------------------------------------------
// Weight gradients. Both operands are [tokens, features] row-major and the MFMA needs eight consecutive tokens of one feature
// per lane from each, so 64-token chunks of both slabs pass through registers into one of two LDS buffers (rows padded by 64
// bytes: the four rows and pieces a 16-lane group of a transposed read touches fall on distinct banks) while the chunk before is
// multiplied, and both fragments are read with ds_read_b64_tr_b16. A workgroup owns a TN x TK tile of one layer's gradient over its
// share of the tokens; all tiles of all layers form one launch of about one workgroup per compute unit (two of the 128 x 128 tiles;
// a workgroup of the large ones fills one with its LDS), so a block's partial sums are one chip's worth of tiles (64 MB at D = 256)
// instead of one per layer.
// Bound: HBM - the operands are read once per 256 features of the other side.
// ------------------------------------------------------------------------------------------------------------------
constexpr int kChunk = 64;
constexpr int kXcds = 8;

struct WgradParams {
  WgradItem item[kWgradItems];
  int32_t first_tile[kWgradItems + 1];
  float* partial;          // per item [splits][N][K], items one behind the other
  float* bias_partial;     // per item [splits][N]
  int64_t partial_at[kWgradItems], bias_at[kWgradItems];
  const int32_t* count;
  int64_t M;
  int32_t splits, n_items;
};

template <int TN, int TK, int WN, int WK>
__global__ __launch_bounds__(WN * WK * kWave, 2) void wgrad_block_kernel(const WgradParams p) {
  constexpr int THREADS = WN * WK * kWave;
  constexpr int BN = TN / WN / 32, BK = TK / WK / 32;   // 32 x 32 blocks of a wavefront
  constexpr int ROWN = TN * 2 + 64, ROWK = TK * 2 + 64;  // LDS row bytes
  constexpr int SLABN = kChunk * ROWN, SLABK = kChunk * ROWK;
  constexpr int PN = kChunk * (TN / 8) / THREADS, PK = kChunk * (TK / 8) / THREADS;  // 16-byte pieces per thread and chunk
  constexpr int RN = THREADS / (TN / 8), RK = THREADS / (TK / 8);                    // rows between a thread's pieces
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  // Workgroups are handed to the eight XCDs in turn; the tiles of a split, which read the same rows, go to one XCD and meet in its L2.
  const int tiles = p.first_tile[p.n_items];
  const int n_wg = static_cast<int>(gridDim.x), xcd = static_cast<int>(blockIdx.x) % kXcds, slot = static_cast<int>(blockIdx.x) / kXcds;
  const int unit = xcd * (n_wg / kXcds) + (xcd < n_wg % kXcds ? xcd : n_wg % kXcds) + slot;
  const int tile = unit % tiles, split = unit / tiles;
  int which = 0;
#pragma unroll
  for (int i = 1; i < kWgradItems; ++i)
    if (i < p.n_items && tile >= p.first_tile[i]) which = i;
  const WgradItem& it = p.item[which];
  const int N = it.N, K = it.K;
  const int tiles_k = (K + TK - 1) / TK;
  const int local = tile - p.first_tile[which];
  const int n0 = (local / tiles_k) * TN, k0 = (local % tiles_k) * TK;
  int64_t rows = p.M;
  {
    const int64_t n = *p.count;
    rows = n < rows ? n : rows;
  }
  const int64_t per = ((rows + p.splits - 1) / p.splits + kChunk - 1) / kChunk * kChunk;
  const int64_t m_begin = split * per;
  const int64_t m_end = m_begin + per < rows ? m_begin + per : rows;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int wn = wave / WK, wk = wave % WK;
  const int g = lane / 16, r = lane % 16;
  const uint32_t a_lane = static_cast<uint32_t>((8 * (g / 2) + r / 4) * ROWN + (16 * (g % 2) + 4 * (r % 4)) * 2 + wn * (TN / WN) * 2);
  const uint32_t b_lane = static_cast<uint32_t>(SLABN + (8 * (g / 2) + r / 4) * ROWK + (16 * (g % 2) + 4 * (r % 4)) * 2 + wk * (TK / WK) * 2);

  f32x16 acc[BN][BK];
#pragma unroll
  for (int i = 0; i < BN; ++i)
#pragma unroll
    for (int j = 0; j < BK; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // a thread's pieces: always the same eight columns, rows tid / (T / 8) + R * i
  const int rn = tid / (TN / 8), cn = n0 + tid % (TN / 8) * 8;
  const int rk = tid / (TK / 8), ck = k0 + tid % (TK / 8) * 8;
  const bool n_ok = cn < N, k_ok = ck < K;
  // (a chunk of kChunk tokens lies in one row block of the panel order, a piece of eight columns in one panel)
  static_assert(kPanelRows % kChunk == 0 && kPanelCols % 8 == 0, "chunks and pieces do not straddle panels");
  auto column = [](int c, bool panels) -> int64_t { return panels ? c / kPanelCols * kPanel + c % kPanelCols : c; };
  const bf16_t* dy_col = it.dy + column(n_ok ? cn : 0, it.dy_panels);
  const bf16_t* a_col = it.a + column(k_ok ? ck : 0, it.a_panels);
  const int64_t dy_ld = it.dy_panels ? kPanelCols : N, a_ld = it.a_panels ? kPanelCols : K;
  const float* rscale = it.scale;
  u32x4 va[PN], vb[PK];
  float sb[PK];
  const u32x4 zero = {0u, 0u, 0u, 0u};
  auto fetch = [&](int64_t m0) {
    const bf16_t* dy_chunk = dy_col + (it.dy_panels ? panel_row(m0, N) : m0 * N);
    const bf16_t* a_chunk = a_col + (it.a_panels ? panel_row(m0, K) : m0 * K);
#pragma unroll
    for (int i = 0; i < PN; ++i) {
      const int64_t m = m0 + rn + RN * i;
      va[i] = (m < m_end && n_ok) ? *reinterpret_cast<const u32x4*>(dy_chunk + (rn + RN * i) * dy_ld) : zero;
    }
#pragma unroll
    for (int i = 0; i < PK; ++i) {
      const int64_t m = m0 + rk + RK * i;
      const bool ok = m < m_end && k_ok;
      vb[i] = ok ? *reinterpret_cast<const u32x4*>(a_chunk + (rk + RK * i) * a_ld) : zero;
      sb[i] = (ok && rscale != nullptr) ? rscale[m] : 1.f;
    }
  };
  if (m_begin < m_end) fetch(m_begin);
  const bool with_bias = it.db != nullptr && k0 == 0;
  float csum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  for (int64_t m0 = m_begin; m0 < m_end; m0 += kChunk) {
    // the buffer written now was last read two chunks ago; the barrier of the chunk in between lies behind those reads
    uint8_t* stage = smem + buf * (SLABN + SLABK);
    if (with_bias) {
#pragma unroll
      for (int i = 0; i < PN; ++i)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          csum[2 * w] += __uint_as_float(va[i][w] << 16);
          csum[2 * w + 1] += __uint_as_float(va[i][w] & 0xffff0000u);
        }
    }
#pragma unroll
    for (int i = 0; i < PN; ++i) *reinterpret_cast<u32x4*>(stage + (rn + RN * i) * ROWN + (cn - n0) * 2) = va[i];
#pragma unroll
    for (int i = 0; i < PK; ++i) {
      if (rscale != nullptr) {
        bf16x8 v = __builtin_bit_cast(bf16x8, vb[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) * sb[i]);
        vb[i] = __builtin_bit_cast(u32x4, v);
      }
      *reinterpret_cast<u32x4*>(stage + SLABN + (rk + RK * i) * ROWK + (ck - k0) * 2) = vb[i];
    }
    if (m0 + kChunk < m_end) fetch(m0 + kChunk);
    __syncthreads();
    const uint32_t base = lds_offset(stage);
    static_for<kChunk / 16>([&](auto ks_tag) {
      constexpr int ks = decltype(ks_tag)::value;
      u32x2 fa[BN][2], fb[BK][2];
      static_for<BN>([&](auto t_tag) {
        constexpr int t = decltype(t_tag)::value;
        lds_read_tr16<(ks * 16) * ROWN + t * 64>(fa[t][0], base + a_lane);
        lds_read_tr16<(ks * 16 + 4) * ROWN + t * 64>(fa[t][1], base + a_lane);
      });
      static_for<BK>([&](auto t_tag) {
        constexpr int t = decltype(t_tag)::value;
        lds_read_tr16<(ks * 16) * ROWK + t * 64>(fb[t][0], base + b_lane);
        lds_read_tr16<(ks * 16 + 4) * ROWK + t * 64>(fb[t][1], base + b_lane);
      });
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[0][0]), "+v"(fa[0][1]) : : "memory");
#pragma unroll
      for (int t = 0; t < BN; ++t) asm volatile("" : "+v"(fa[t][0]), "+v"(fa[t][1]));
#pragma unroll
      for (int t = 0; t < BK; ++t) asm volatile("" : "+v"(fb[t][0]), "+v"(fb[t][1]));
#pragma unroll
      for (int i = 0; i < BN; ++i)
#pragma unroll
        for (int j = 0; j < BK; ++j) {
          const u32x4 abits = {fa[i][0][0], fa[i][0][1], fa[i][1][0], fa[i][1][1]};
          const u32x4 bbits = {fb[j][0][0], fb[j][0][1], fb[j][1][0], fb[j][1][1]};
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, abits), __builtin_bit_cast(bf16x8, bbits),
                                                              acc[i][j], 0, 0, 0);
        }
    });
    buf ^= 1;
  }
  float* out = p.partial + p.partial_at[which] + static_cast<int64_t>(split) * N * K;
  const int l32 = lane % 32, hh = lane / 32;
#pragma unroll
  for (int i = 0; i < BN; ++i)
#pragma unroll
    for (int j = 0; j < BK; ++j) {
      const int col = k0 + wk * (TK / WK) + j * 32 + l32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = n0 + wn * (TN / WN) + i * 32 + (e / 4) * 8 + hh * 4 + (e % 4);
        if (row < N && col < K) out[static_cast<int64_t>(row) * K + col] = acc[i][j][e];
      }
    }
  if (with_bias) {
    __syncthreads();  // every wavefront is done with the chunk buffers
    float* red = reinterpret_cast<float*>(smem);  // [RN row groups][TN columns]
#pragma unroll
    for (int e = 0; e < 8; ++e) red[rn * TN + (cn - n0) + e] = csum[e];
    __syncthreads();
    for (int c = tid; c < TN; c += THREADS) {
      if (n0 + c >= N) continue;
      float sum = 0.f;
#pragma unroll
      for (int rg = 0; rg < RN; ++rg) sum += red[rg * TN + c];
      p.bias_partial[p.bias_at[which] + static_cast<int64_t>(split) * N + n0 + c] = sum;
    }
  }
}

// dw = sum of the splits, in order, times the norm's weight per column; per workgroup of kReduceRows rows the column sums of
// w * G (the gradient of the norm's weight) are left in norm_partial [row blocks][K].
constexpr int kReduceThreads = 256;
constexpr int kReduceRows = 16;
struct ReduceParams {
  WgradItem item[kWgradItems];
  int32_t first_unit[kWgradItems + 1];   // workgroups: row blocks x column blocks of an item
  const float* partial;
  int64_t partial_at[kWgradItems];
  float* norm_partial;
  int64_t norm_at[kWgradItems];
  int32_t splits, n_items;
};
template <typename T>
__global__ __launch_bounds__(kReduceThreads) void wgrad_reduce_kernel(const ReduceParams p) {
  __shared__ f32x4 red[4][kWave];
  int which = 0;
#pragma unroll
  for (int i = 1; i < kWgradItems; ++i)
    if (i < p.n_items && static_cast<int>(blockIdx.x) >= p.first_unit[i]) which = i;
  const WgradItem& it = p.item[which];
  const int N = it.N, K = it.K;
  const int col_blocks = (K + 255) / 256;
  const int local = static_cast<int>(blockIdx.x) - p.first_unit[which];
  const int row0 = local / col_blocks * kReduceRows;
  const int col = local % col_blocks * 256 + static_cast<int>(threadIdx.x % kWave) * 4;  // K is a multiple of 8
  const int rg = threadIdx.x / kWave;
  const int64_t nk = static_cast<int64_t>(N) * K;
  const float* src = p.partial + p.partial_at[which];
  f32x4 nw = {1.f, 1.f, 1.f, 1.f}, nsum = {0.f, 0.f, 0.f, 0.f};
  const bool ok = col < K;
  if (ok && it.norm_w != nullptr)
#pragma unroll
    for (int e = 0; e < 4; ++e) nw[e] = static_cast<float>(static_cast<const T*>(it.norm_w)[col + e]);
#pragma unroll
  for (int i = 0; i < kReduceRows / 4; ++i) {
    const int row = row0 + rg + 4 * i;
    if (!ok || row >= N) continue;
    const int64_t at = static_cast<int64_t>(row) * K + col;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < p.splits; k += 8) {  // eight partials requested at once, added in order
      f32x4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const f32x4*>(src + (k + j < p.splits ? k + j : k) * nk + at);
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += k + j < p.splits ? v[j][e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (it.dnorm != nullptr) nsum[e] = fmaf(s[e], static_cast<float>(static_cast<const T*>(it.w)[at + e]), nsum[e]);
      static_cast<T*>(it.dw)[at + e] = static_cast<T>(s[e] * nw[e]);
    }
  }
  if (it.dnorm == nullptr) return;  // the same for the whole workgroup
  red[rg][threadIdx.x % kWave] = nsum;
  __syncthreads();
  if (rg == 0 && ok) {
#pragma unroll
    for (int w = 1; w < 4; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) nsum[e] += red[w][threadIdx.x][e];
    *reinterpret_cast<f32x4*>(p.norm_partial + p.norm_at[which] + static_cast<int64_t>(row0 / kReduceRows) * K + col) = nsum;
  }
}

constexpr int kVectorItems = 64;
struct VectorParams {
  VectorItem item[kVectorItems];
  int32_t first_unit[kVectorItems + 1];
  int32_t n;
};
// 16 columns per workgroup, 16 slices of the partial rows: slice sums in row order, added in slice order.
template <typename T>
__global__ __launch_bounds__(256) void sum_vectors_kernel(const VectorParams p) {
  __shared__ float red[16][16];
  int which = 0;
  for (int lo = 0, hi = p.n; lo < hi;) {  // last item whose first unit is not above this one
    const int mid = (lo + hi) / 2;
    if (p.first_unit[mid] <= static_cast<int>(blockIdx.x)) {
      which = mid;
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  const VectorItem& it = p.item[which];
  const int c = (static_cast<int>(blockIdx.x) - p.first_unit[which]) * 16 + static_cast<int>(threadIdx.x % 16);
  const int slice = threadIdx.x / 16;
  float sum = 0.f;
  if (c < it.cols) {
    constexpr int kAhead = 8;  // rows requested together, added in their order: one by one each is a memory latency (31 -> 8 us, four blocks of width 256 at 1024 x 512 positions)
    int i = slice;
    for (; i + 16 * (kAhead - 1) < it.parts; i += 16 * kAhead) {
      float v[kAhead];
#pragma unroll
      for (int a = 0; a < kAhead; ++a) v[a] = it.src[static_cast<int64_t>(i + 16 * a) * it.stride + c];
#pragma unroll
      for (int a = 0; a < kAhead; ++a) sum += v[a];
    }
    for (; i < it.parts; i += 16) sum += it.src[static_cast<int64_t>(i) * it.stride + c];
  }
  red[slice][threadIdx.x % 16] = sum;
  __syncthreads();
  if (slice == 0 && c < it.cols) {
    float total = 0.f;
#pragma unroll
    for (int sl = 0; sl < 16; ++sl) total += red[sl][threadIdx.x];
    static_cast<T*>(it.dst)[c] = static_cast<T>(total);
  }
}

// 256 x 256 tiles where the layers are that wide and the batch fills the chip with them; 128 x 128 tiles of four wavefronts, two
// workgroups per compute unit, for the narrow model and for small batches: there a tile's chain over its chunks and its store are the
// time, not the operands, which L2 holds, and four times as many tiles need fewer splits and partial sums. Gradients and their
// reduction, us per block, 256- / 128-wide tiles, F = 1024 (F = 512), by positions of which 6 in 10 hold tokens: 1 024 50 / 27,
// 3 216 39 / 28, 9 648 49 / 42 (45 / 36), 15 360 (48 / 46), 16 384 58 / 59 (49 / 47); from 42 496 on the step is 1 - 7 % slower.
// At least 512 tokens a split: with 1 024 it is 37 instead of 27 at 1 024 positions and, D = 128, 35 instead of 25; 256 lies within 4 us
// either way.
struct WgradPlan {
  int tn, tk, tiles, splits;
};
WgradPlan plan_of(int64_t M, const int32_t (*shapes)[2], int items) {
  WgradPlan pl{};
  int min_side = 1 << 30;
  for (int i = 0; i < items; ++i) min_side = shapes[i][0] < min_side ? shapes[i][0] : (shapes[i][1] < min_side ? shapes[i][1] : min_side);
  const int cus = compute_units() > 0 ? compute_units() : 1;
  pl.tn = pl.tk = min_side >= 256 && M >= 64 * static_cast<int64_t>(cus) ? 256 : 128;
  for (int i = 0; i < items; ++i) pl.tiles += ((shapes[i][0] + pl.tn - 1) / pl.tn) * ((shapes[i][1] + pl.tk - 1) / pl.tk);
  // about one workgroup per compute unit (two of the small ones), but no split of fewer than 512 tokens: a split costs a pass
  // over its partial tile
  const int want = (pl.tn == 256 ? 1 : 2) * cus / pl.tiles;
  const int64_t most = (M + 511) / 512;
  pl.splits = want < 1 ? 1 : want;
  if (pl.splits > most) pl.splits = most < 1 ? 1 : static_cast<int>(most);
  return pl;
}

}  // namespace

int dgrad_norm(const char* name, const void* dy, bool dy_panels, int32_t K, const void* w_t, const void* x, const float* rstd, const void* norm_w,
               const void* dres, void* dx, int64_t M, int32_t D, const int32_t* count, hipStream_t s) {
  DgradParams p{};
  p.dy = static_cast<const bf16_t*>(dy);
  p.w_t = static_cast<const bf16_t*>(w_t);
  p.x = static_cast<const bf16_t*>(x);
  p.rstd = rstd;
  p.norm_w = static_cast<const bf16_t*>(norm_w);
  p.dres = static_cast<const bf16_t*>(dres);
  p.dx = static_cast<bf16_t*>(dx);
  p.count = count;
  p.M = M;
  p.K = K;
  p.panels = dy_panels;
  const int cus = compute_units();
  const bool small = M < 128 * static_cast<int64_t>(cus);
  // Two 128-token workgroups share a compute unit, so that one's epilogue runs beside the other's products: worth the second pass
  // over the weights where the contraction is short, and where 256-token workgroups would be less than two rounds (294 912
  // tokens, D = 256, 128- / 256-token workgroups: K = 768 207 / 222 us, K = 2048 420 / 400; 51 584 rows: 347 / 430 us over both).
  if (small) return D == 256 ? launch_dgrad<256, 1, 8, 64, 3>(p, s, name) : launch_dgrad<128, 1, 4, 64, 3>(p, s, name);
  if (D == 128) return launch_dgrad<128, 4, 2, 32, 4>(p, s, name);
  if (K <= 1024 || M < 512 * static_cast<int64_t>(cus)) return launch_dgrad<256, 2, 2, 32, 3>(p, s, name);
  return launch_dgrad<256, 4, 2, 32, 4>(p, s, name);
}

int64_t wgrad_scratch_floats(int64_t M, const int32_t (*shapes)[2], int items) {
  const WgradPlan pl = plan_of(M, shapes, items);
  int64_t n = 0;
  for (int i = 0; i < items; ++i) n += static_cast<int64_t>(pl.splits) * shapes[i][0] * shapes[i][1];
  return n;
}

int64_t wgrad_vector_floats(int64_t M, const int32_t (*shapes)[2], int items) {
  const WgradPlan pl = plan_of(M, shapes, items);
  int64_t n = 0;
  for (int i = 0; i < items; ++i)
    n += static_cast<int64_t>(pl.splits) * shapes[i][0] + static_cast<int64_t>((shapes[i][0] + kReduceRows - 1) / kReduceRows) * shapes[i][1];
  return n;
}

int wgrad_block(const char* name, const WgradItem* items, int n_items, int64_t M, const int32_t* count, float* scratch,
                float* vectors, int dtype, VectorItem* out_vectors, int* n_vectors, hipStream_t s) {
  int32_t shapes[kWgradItems][2];
  for (int i = 0; i < n_items; ++i) {
    shapes[i][0] = items[i].N;
    shapes[i][1] = items[i].K;
  }
  const WgradPlan pl = plan_of(M, shapes, n_items);
  WgradParams p{};
  ReduceParams q{};
  int tiles = 0, units = 0;
  int64_t at = 0, vec = 0;
  for (int i = 0; i < n_items; ++i) {
    const WgradItem& it = items[i];
    p.item[i] = q.item[i] = it;
    p.first_tile[i] = tiles;
    tiles += ((it.N + pl.tn - 1) / pl.tn) * ((it.K + pl.tk - 1) / pl.tk);
    p.partial_at[i] = q.partial_at[i] = at;
    at += static_cast<int64_t>(pl.splits) * it.N * it.K;
    p.bias_at[i] = vec;
    if (it.db != nullptr) out_vectors[(*n_vectors)++] = VectorItem{vectors + vec, it.db, pl.splits, it.N, it.N};
    vec += static_cast<int64_t>(pl.splits) * it.N;
    const int row_blocks = (it.N + kReduceRows - 1) / kReduceRows;
    q.first_unit[i] = units;
    units += row_blocks * ((it.K + 255) / 256);
    q.norm_at[i] = vec;
    if (it.dnorm != nullptr) out_vectors[(*n_vectors)++] = VectorItem{vectors + vec, it.dnorm, row_blocks, it.K, it.K};
    vec += static_cast<int64_t>(row_blocks) * it.K;
  }
  p.first_tile[n_items] = tiles;
  q.first_unit[n_items] = units;
  p.partial = scratch;
  p.bias_partial = vectors;
  p.count = count;
  p.M = M;
  p.splits = q.splits = pl.splits;
  p.n_items = q.n_items = n_items;
  q.partial = scratch;
  q.norm_partial = vectors;
  const dim3 grid(tiles * pl.splits);
  auto go = [&](auto kernel, int threads, size_t lds) -> int {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) !=
        hipSuccess)
      return set_error(TAAC_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", name, lds);
    hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, s, p);
    return check_launch(name);
  };
  const size_t lds = 2 * 2 * static_cast<size_t>(kChunk) * (pl.tn * 2 + 64);
  const int rc = pl.tn == 256 ? go(wgrad_block_kernel<256, 256, 2, 4>, 512, lds) : go(wgrad_block_kernel<128, 128, 2, 2>, 256, lds);
  if (rc != TAAC_OK) return rc;
  if (dtype == TAAC_F32)
    hipLaunchKernelGGL(wgrad_reduce_kernel<float>, dim3(units), dim3(kReduceThreads), 0, s, q);
  else
    hipLaunchKernelGGL(wgrad_reduce_kernel<bf16_t>, dim3(units), dim3(kReduceThreads), 0, s, q);
  return check_launch(name);
}

int sum_vectors(const char* name, const VectorItem* items, int n, int dtype, hipStream_t s) {
  for (int base = 0; base < n; base += kVectorItems) {
    VectorParams p{};
    p.n = n - base < kVectorItems ? n - base : kVectorItems;
    int units = 0;
    for (int i = 0; i < p.n; ++i) {
      p.item[i] = items[base + i];
      p.first_unit[i] = units;
      units += (items[base + i].cols + 15) / 16;
    }
    if (dtype == TAAC_F32)
      hipLaunchKernelGGL(sum_vectors_kernel<float>, dim3(units), dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL(sum_vectors_kernel<bf16_t>, dim3(units), dim3(256), 0, s, p);
    const int rc = check_launch(name);
    if (rc != TAAC_OK) return rc;
  }
  return TAAC_OK;
}

}  // namespace taac
