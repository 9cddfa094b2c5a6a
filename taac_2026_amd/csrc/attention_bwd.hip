// Backward of the key-length-masked attention for gfx950 (head dims up to 64, bf16 / fp16 storage, fp32 arithmetic).
//
// With S = Q K^T / sqrt(d), P = exp(S - lse) (lse saved by the training forward), D_i = sum_d O[i, d] dO[i, d]:
//   dV = P^T dO,   dP = dO V^T,   dS = P * (dP - D) / sqrt(d),   dQ = dS K,   dK = dS^T Q
// (the recipe of the reference's backward kernels, accelerators/attention/kernels/tilelang.py:405-435, 598-699).
// Every output element has exactly one writer and a fixed summation order (the reference accumulates dQ with
// floating-point atomics). Where a workgroup can hold a sample's keys, attn_bwd_fused_kernel forms all three gradients
// at once; otherwise two kernels, both recomputing S and dP from the inputs:
//   attn_bwd_dq_kernel   one workgroup per (batch, head, 128 queries): a lane owns one query, the keys stream through
//                        LDS in chunks of 64; also writes D for the second kernel.
//   attn_bwd_dkv_kernel  one workgroup per (batch, head, 128 keys): a lane owns one key, the queries stream through LDS.
// All products are formed transposed, as in the forward kernel: the streamed operand is the MFMA A operand (rows from
// LDS), the lane-owned operand the B operand (registers), so the accumulator holds one owned column per lane and the
// 16 registers run over the streamed rows (register r <-> row (r / 4) * 8 + hh * 4 + r % 4 of a 32-row tile). The
// second product of each pair consumes those values as a B operand; its streamed A operand is the same chunk read
// column-wise with ds_read_b64_tr_b16, at row offsets that follow that register order, so every chunk is staged once,
// row-major, and nothing is transposed on the way into LDS.
#include <math.h>

#include "ts_common.h"

namespace taac {
namespace {

constexpr int kThreads = 256;
constexpr int kOwn = 128;    // owned rows (queries or keys) per workgroup: 32 per wavefront
constexpr int kChunk = 64;   // streamed rows per LDS chunk

struct AttnBwdParams {
  const void* q;
  const void* k;
  const void* v;
  const void* o;
  const void* dout;
  const float* lse;       // [B, H, Tq]
  float* delta;           // [B, H, Tq] workspace: written by the dQ kernel, read by the dK / dV kernel
  void* dq;
  void* dk;
  void* dv;
  const int32_t* key_lengths;
  const uint8_t* drop_mask;  // byte mask with rows [Tq][Tk] at batch / head strides mask_bs / mask_hs, or null:
                             // training dropout (keep mask, non-zero = keep) or pair visibility (non-zero = visible)
  int64_t mask_bs, mask_hs;  // elements between the mask matrices of consecutive samples / heads (0: shared)
  const uint8_t* key_valid;  // visibility mode: [B, Tk] bytes, non-zero = the key can be seen at all; or null
                             // (bit modes: [B, ceil(Tk / 32)] words)
  const uint32_t* bit_words; // bit modes: rows of ceil(Tk / 32) words per query, bits_bs words between the samples' matrices
  int64_t bits_bs;
  float drop_scale;          // 1 / (1 - p)
  int32_t B, H, Tq, Tk, d;
  int64_t qs[4], ks[4], vs[4], os[4], dos[4], dqs[4], dks[4], dvs[4];
  const int32_t* row_offsets;  // sample b's rows start at row row_offsets[b] of every tensor (a compact tensor of the batch's valid
                               // tokens: rows at or beyond the length belong to the next sample and are not written), or null
  float scale;            // 1 / sqrt(d)
  int32_t zero_pad;       // query rows at or beyond key_lengths[b] carry no gradient
  int32_t causal;
  uint32_t nblk;          // owned-row blocks per (batch, head)
  uint32_t total;
};

// First row of (sample b, head h).
template <bool COMPACT, typename T>
__device__ __forceinline__ T* head_rows(T* base, const int64_t (&strides)[4], const AttnBwdParams& p, int b, int h) {
  const int64_t row0 = COMPACT ? p.row_offsets[b] * strides[2] : b * strides[0];
  return base + row0 + h * strides[1];
}

template <typename T>
struct Mfma32;
template <>
struct Mfma32<bf16_t> {
  static __device__ __forceinline__ f32x16 run(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma32<f16_t> {
  static __device__ __forceinline__ f32x16 run(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

__device__ __forceinline__ float pair_sum(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) + __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

template <typename T>
__device__ __forceinline__ uint32_t pack2(T lo, T hi) {
  return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, lo)) |
         (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, hi)) << 16);
}

// A streamed chunk (kChunk rows of DP features) lies row-major and unpadded in LDS, the 16-byte pieces of row r stored
// at piece ^ row_swizzle(r), and serves two kinds of reads without bank conflicts:
//   rows as MFMA A operands (lane l32 reads one piece of row l32: 16 consecutive rows of one piece cover all banks);
//   columns as MFMA A operands through ds_read_b64_tr_b16: a 16-lane group reads 32 contiguous bytes of four
//   consecutive rows and every lane receives four rows of one feature (see streamed_column_offset below).
// +32 rows leave the swizzle unchanged, +16 rows too, +8 rows flip SwizzleStep::kRows8 of the address. Four rows further it is another
// pair of pieces, for the transposed reads of eight consecutive rows (attn_bwd_fused_kernel's dQ).
template <int DP>
__device__ __forceinline__ int row_swizzle(int r) {
  static_assert(DP == 32 || DP == 64, "row swizzles are written for 64- and 128-byte rows");
  return DP == 32 ? ((r >> 1) & 2) | ((r >> 3) & 1) : ((r >> 1) & 7) ^ (((r >> 1) & 1) << 2);
}
template <int DP>
struct SwizzleStep {
  static constexpr uint32_t kRows8 = (DP == 32 ? 1 : 4) * 16;  // address bits that +8 rows flip
};

// Staging of one streamed operand. DMA: the chunk goes from global memory straight into LDS (one 1 KB transfer per
// wavefront and piece slot, no staging registers); rows at or beyond row_end repeat the last valid row, whose products
// the callers cancel (finite values times a zero probability); needs d == DP and 32-bit source offsets. Otherwise the
// chunk travels through registers (fetch, then commit after the barrier), with zeros for rows at or beyond row_end and
// features at or beyond d. The lane's slot i * 256 + tid is (row slot / C8, stored piece slot % C8).
template <typename T, int DP, bool DMA>
struct Streamed {
  typedef typename Vec8<T>::type vec_t;
  static constexpr int C8 = DP / 8, ROWB = DP * 2, TILE_BYTES = kChunk * ROWB;
  static constexpr int PPT = kChunk * C8 / kThreads;
  static_assert(kChunk * C8 % kThreads == 0, "whole transfers per wavefront");
  const T* base;
  int64_t stride;
  int srow, piece;          // the lane's row inside a chunk (slot 0) and the logical piece stored at its slot
  uint32_t row_bytes;
  vec_t reg[DMA ? 1 : PPT];
  __device__ __forceinline__ void init(const T* b, int64_t st, int tid) {
    base = b;
    stride = st;
    srow = tid / C8;
    piece = (tid % C8) ^ row_swizzle<DP>(srow);
    row_bytes = static_cast<uint32_t>(st) * 2u;
  }
  __device__ __forceinline__ void fetch(int row0, int row_end, int d, uint8_t* tile, int tid) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      int row = row0 + srow + i * (kThreads / C8);
      if (DMA) {
        row = row < row_end ? row : row_end - 1;  // row_end >= 1 here
        lds_dma16_offset(base, __umul24(static_cast<uint32_t>(row), row_bytes) + static_cast<uint32_t>(piece * 16),
                         tile + i * (kThreads * 16) + (tid / kWave) * (kWave * 16));
      } else if (row < row_end && piece * 8 < d) {
        reg[DMA ? 0 : i] = *reinterpret_cast<const vec_t*>(base + row * stride + piece * 8);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) reg[DMA ? 0 : i][e] = static_cast<T>(0.f);
      }
    }
  }
  __device__ __forceinline__ void commit(uint8_t* tile, int tid) const {
    if (DMA) return;
#pragma unroll
    for (int i = 0; i < PPT; ++i) *reinterpret_cast<vec_t*>(tile + i * (kThreads * 16) + tid * 16) = reg[DMA ? 0 : i];
  }
};

// Byte offset (inside a chunk tile) of the lane's row fragment of k-step 0 of a 32-row tile: row l32, piece hh; k-step s
// is this offset with s * 32 XORed in, the next 32-row tile 32 * ROWB further.
template <int DP>
__device__ __forceinline__ uint32_t streamed_row_offset(int l32, int hh) {
  return static_cast<uint32_t>(l32 * (DP * 2) + ((hh ^ row_swizzle<DP>(l32)) * 16));
}

// Byte offset of the lane's address for the transposed reads. Accumulator register j of a 32-row tile belongs to row
// (j / 4) * 8 + hh * 4 + j % 4, so the B operand of the second product (registers 8 s2 .. 8 s2 + 7) runs over rows
// 16 s2 + hh * 4 + 0..3 and 16 s2 + 8 + hh * 4 + 0..3. The matching A operand holds, for feature l32 (of row block mb),
// those eight rows: two transposed reads, at row offsets 16 s2 and 16 s2 + 8, in each of which lane r of 16-lane group
// g points at row hh * 4 + r / 4, features 16 (g % 2) + 4 (r % 4) .. + 3. Row block mb XORs 64 mb into the offset and
// the read 8 rows further SwizzleStep<DP>::kRows8.
template <int DP>
__device__ __forceinline__ uint32_t streamed_column_offset(int lane) {
  const int row = 4 * (lane / 32) + (lane % 16) / 4;
  const int piece = 2 * ((lane / 16) % 2) + (lane % 4) / 2;
  return static_cast<uint32_t>(row * (DP * 2) + ((piece ^ row_swizzle<DP>(row)) * 16) + (lane % 2) * 8);
}

// A operand of the second product for (32-row tile at byte offset tile_off, k-step s2) from a tile base address.
template <typename T, int DP, int TILE_OFF>
__device__ __forceinline__ void read_columns(u32x2 (&frag)[2], uint32_t addr) {
  lds_read_tr16<TILE_OFF>(frag[0], addr);
  lds_read_tr16<TILE_OFF + 8 * DP * 2>(frag[1], addr ^ SwizzleStep<DP>::kRows8);
}

// Owned rows as B-operand fragments: lane (l32, hh) holds features 16 s + 8 hh .. + 7 of row `row` (zeros when !ok).
template <typename T, int DP>
__device__ __forceinline__ void load_owned(const T* __restrict__ base, int64_t stride, int row, bool ok, int d, int hh,
                                           typename Vec8<T>::type (&frag)[DP / 16]) {
  typedef typename Vec8<T>::type vec_t;
#pragma unroll
  for (int s = 0; s < DP / 16; ++s) {
    const int col = 16 * s + 8 * hh;
    if (ok && col < d) {
      frag[s] = *reinterpret_cast<const vec_t*>(base + row * stride + col);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) frag[s][e] = static_cast<T>(0.f);
    }
  }
}

// Writes MB accumulators (transposed tile: rows = features, column = owned row of the lane) as rows of `out`.
template <typename T, int DP>
__device__ __forceinline__ void store_owned(const f32x16 (&acc)[DP / 32], uint8_t* tile, T* __restrict__ out,
                                            int64_t stride, int row0, int row_limit, int d, int lane) {
  typedef typename Vec8<T>::type vec_t;
  typedef typename Vec8<T>::half_type vec4_t;
  constexpr int C8 = DP / 8, OROW = DP * 2 + 16;
  const int l32 = lane % 32, hh = lane / 32;
#pragma unroll
  for (int mb = 0; mb < DP / 32; ++mb)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      vec4_t ov;
#pragma unroll
      for (int e = 0; e < 4; ++e) ov[e] = static_cast<T>(acc[mb][jq * 4 + e]);
      *reinterpret_cast<vec4_t*>(tile + l32 * OROW + (mb * 32 + jq * 8 + hh * 4) * 2) = ov;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int RPP = kWave / C8;
  const int c8 = lane % C8;
#pragma unroll
  for (int pass = 0; pass < 32 / RPP; ++pass) {
    const int r = pass * RPP + lane / C8;
    const vec_t val = *reinterpret_cast<const vec_t*>(tile + r * OROW + c8 * 16);
    if (row0 + r < row_limit && c8 * 8 < d) *reinterpret_cast<vec_t*>(out + (row0 + r) * stride + c8 * 8) = val;
  }
}

// A transposed read (lds_read_tr16) that the compiler waits for.
template <typename T>
__device__ __forceinline__ typename Vec8<T>::half_type read_tr16(uint32_t addr) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  return __builtin_bit_cast(typename Vec8<T>::half_type, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_ptr>(addr)));
}

// The fragments of read_columns, awaited by the compiler.
template <typename T, int DP>
__device__ __forceinline__ void fetch_columns(typename Vec8<T>::half_type (&frag)[2][2], uint32_t addr) {
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    frag[s2][0] = read_tr16<T>(addr + s2 * (16 * DP * 2));
    frag[s2][1] = read_tr16<T>((addr ^ SwizzleStep<DP>::kRows8) + s2 * (16 * DP * 2) + 8 * DP * 2);
  }
}

template <typename H>
__device__ __forceinline__ auto join(H lo, H hi) {
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// `value` where bit `at` of the word is set (bits: 1), else zero, in two instructions: a signed one-bit field is all ones or nothing.
// (Masked blocks of 128 x 403 tokens, 8 heads of 32: dK / dV kernel 67.4 -> 62.5 us. dQ's waits for words that were requested right in front
// of the wait cost it as much: 66.3 -> 62.2.)
__device__ __forceinline__ float where_bit(float value, uint32_t word, int at, int bits) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, value) & static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(word), at, bits)));
}

// The second product of a 32-row tile: acc[mb] += columns(tile)^T-fragments x b[s2], the column fragments read
// transposed from the chunk tile at `addr` (tile base + streamed_column_offset), one row block at a time.
template <typename T, int DP, int TILE_OFF>
__device__ __forceinline__ void accumulate_columns(f32x16 (&acc)[DP / 32], const typename Vec8<T>::type (&b)[2], uint32_t addr) {
  typedef typename Vec8<T>::type vec_t;
  static_for<DP / 32>([&](auto mb_tag) {
    constexpr int mb = decltype(mb_tag)::value;
    u32x2 f[2][2];
    read_columns<T, DP, TILE_OFF>(f[0], addr ^ (mb * 64));
    read_columns<T, DP, TILE_OFF + 16 * DP * 2>(f[1], addr ^ (mb * 64));
    // hand-issued reads are awaited by hand; the fragments are tied to the wait so that no consumer moves above it
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0][0]), "+v"(f[0][1]), "+v"(f[1][0]), "+v"(f[1][1]) : : "memory");
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const u32x4 bits = {f[s2][0][0], f[s2][0][1], f[s2][1][0], f[s2][1][1]};
      acc[mb] = Mfma32<T>::run(__builtin_bit_cast(vec_t, bits), b[s2], acc[mb]);
    }
  });
}

// Same for two accumulators that share the tile position (dV from dO and P, dK from Q and dS).
template <typename T, int DP, int TILE_OFF>
__device__ __forceinline__ void accumulate_columns2(f32x16 (&acc_a)[DP / 32], const typename Vec8<T>::type (&b_a)[2],
                                                    uint32_t addr_a, f32x16 (&acc_b)[DP / 32],
                                                    const typename Vec8<T>::type (&b_b)[2], uint32_t addr_b) {
  typedef typename Vec8<T>::type vec_t;
  static_for<DP / 32>([&](auto mb_tag) {
    constexpr int mb = decltype(mb_tag)::value;
    u32x2 fa[2][2], fb[2][2];
    read_columns<T, DP, TILE_OFF>(fa[0], addr_a ^ (mb * 64));
    read_columns<T, DP, TILE_OFF + 16 * DP * 2>(fa[1], addr_a ^ (mb * 64));
    read_columns<T, DP, TILE_OFF>(fb[0], addr_b ^ (mb * 64));
    read_columns<T, DP, TILE_OFF + 16 * DP * 2>(fb[1], addr_b ^ (mb * 64));
    asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(fa[0][0]), "+v"(fa[0][1]), "+v"(fa[1][0]), "+v"(fa[1][1]) : : "memory");
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const u32x4 bits = {fa[s2][0][0], fa[s2][0][1], fa[s2][1][0], fa[s2][1][1]};
      acc_a[mb] = Mfma32<T>::run(__builtin_bit_cast(vec_t, bits), b_a[s2], acc_a[mb]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fb[0][0]), "+v"(fb[0][1]), "+v"(fb[1][0]), "+v"(fb[1][1]) : : "memory");
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const u32x4 bits = {fb[s2][0][0], fb[s2][0][1], fb[s2][1][0], fb[s2][1][1]};
      acc_b[mb] = Mfma32<T>::run(__builtin_bit_cast(vec_t, bits), b_b[s2], acc_b[mb]);
    }
  });
}

// Keep bytes of four consecutive keys of one mask row as one word (byte e = key key0 + e); keys at or beyond Tk read as 0.
__device__ __forceinline__ uint32_t keep_bytes4(const uint8_t* row, int key0, int Tk, bool aligned) {
  if (aligned && key0 + 3 < Tk) return *reinterpret_cast<const uint32_t*>(row + key0);
  uint32_t w = 0u;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (key0 + e < Tk) w |= static_cast<uint32_t>(row[key0 + e]) << (8 * e);
  return w;
}

// MODE (both kernels) says what the byte mask is. kMaskDropout: the caller's keep mask of the training forward; dV takes
// keep ? P / (1 - p) : 0 and the score gradient P * ((keep ? dP / (1 - p) : 0) - D) / sqrt(d), as the reference's backward
// kernel does (tilelang.py:535-570). kMaskVisible: the pairs the forward's mask let through (any bool mask, e.g. a
// structured one written out); an invisible pair has probability 0 - the log-sum-exp was taken over the visible ones.
// kMaskBits: the same as bits, in the layout of the structured forward: drop_mask holds 32-bit words, row i of a sample's
// matrix at word (b * mask_bs + i * wpr), wpr = ceil(Tk / 32), bit j % 32 of word j / 32 = pair (i, j); key_valid holds
// [B, wpr] words. One word per 32-key tile instead of 32 bytes.
// kMaskBitsDropout: the bit form for the pairs AND the byte keep mask of dropout (both pointers).
constexpr int kMaskNone = 0, kMaskDropout = 1, kMaskVisible = 2, kMaskBits = 3, kMaskBitsDropout = 4;

// COMPACT: samples are addressed by row_offsets (decided at run time it costs the other form 1.5 %: every pointer's chain of scalar
// loads stands in front of a workgroup's first rows; 2048 x 4 x 256 x 64: 270 -> 274 and 306 -> 310 us).
template <typename T, int DP, bool DMA, int MODE = kMaskNone, bool COMPACT = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(DP == 32 ? 4 : 3))) void attn_bwd_dq_kernel(const AttnBwdParams p) {
  constexpr bool DROPOUT = MODE == kMaskDropout || MODE == kMaskBitsDropout;
  constexpr bool BITS = MODE == kMaskBits || MODE == kMaskBitsDropout;
  typedef typename Vec8<T>::type vec_t;
  constexpr int KSTEPS = DP / 16, MB = DP / 32;
  constexpr int ROWB = DP * 2, TILE_BYTES = kChunk * ROWB, BUF_BYTES = 2 * TILE_BYTES;  // a chunk of K, then of V
  typedef typename Vec8<T>::half_type vec4_t;
  constexpr bool kAhead = DP == 32 && (MODE == kMaskNone || MODE == kMaskBits);
  constexpr int NBUF = DMA ? 2 : 1;  // direct transfers land in the other buffer while this one is consumed
  constexpr int OROW = DP * 2 + 16;
  constexpr int OUT_BYTES = (kThreads / kWave) * 32 * OROW;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NBUF * BUF_BYTES > OUT_BYTES ? NBUF * BUF_BYTES : OUT_BYTES];

  const uint32_t logical = xcd_remap(blockIdx.x, p.total);
  const int blk = static_cast<int>(logical % p.nblk);
  const int bh = static_cast<int>(logical / p.nblk);
  const int h = bh % p.H, b = bh / p.H;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, l32 = lane % 32, hh = lane / 32;
  const T* qb = head_rows<COMPACT>(static_cast<const T*>(p.q), p.qs, p, b, h);
  const T* kb = head_rows<COMPACT>(static_cast<const T*>(p.k), p.ks, p, b, h);
  const T* vb = head_rows<COMPACT>(static_cast<const T*>(p.v), p.vs, p, b, h);
  const T* ob = head_rows<COMPACT>(static_cast<const T*>(p.o), p.os, p, b, h);
  const T* dob = head_rows<COMPACT>(static_cast<const T*>(p.dout), p.dos, p, b, h);
  T* dqb = head_rows<COMPACT>(static_cast<T*>(p.dq), p.dqs, p, b, h);

  int len = p.Tk;
  if (p.key_lengths != nullptr) {
    len = p.key_lengths[b];
    len = len < 0 ? 0 : (len > p.Tk ? p.Tk : len);
  }
  const int q_valid = p.zero_pad ? (len < p.Tq ? len : p.Tq) : p.Tq;
  const int q_begin = blk * kOwn;
  const int qi = q_begin + wave * 32 + l32;
  const bool q_ok = qi < q_valid;
  int kv_end = len;
  if (p.causal) kv_end = kv_end < q_begin + kOwn ? kv_end : q_begin + kOwn;
  if (q_begin >= q_valid) kv_end = 0;  // a block of padded queries: zero gradient, no key is staged
  // A wavefront whose 32 queries all lie in the padding only helps staging.
  const bool wave_active = q_begin + wave * 32 < q_valid;

  vec_t qf[KSTEPS], dof[KSTEPS], of[KSTEPS];
  load_owned<T, DP>(qb, p.qs[2], qi, q_ok, p.d, hh, qf);
  load_owned<T, DP>(dob, p.dos[2], qi, q_ok, p.d, hh, dof);
  load_owned<T, DP>(ob, p.os[2], qi, q_ok, p.d, hh, of);
  float delta = 0.f;
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) delta = fmaf(static_cast<float>(of[s][e]), static_cast<float>(dof[s][e]), delta);
  delta = pair_sum(delta);
  const int64_t stat = (static_cast<int64_t>(b) * p.H + h) * p.Tq + qi;
  if (hh == 0 && qi < p.Tq) p.delta[stat] = delta;
  const float lse = q_ok ? p.lse[stat] : -INFINITY;
  const float c = p.scale * 1.4426950408889634f;  // scores -> base-2 exponent
  // a row without a visible key (or in the padding) gets +inf: exp2(x - inf) = 0 switches it off without a select
  const float lse2 = lse > -INFINITY ? lse * 1.4426950408889634f : INFINITY;
  const float delta_scaled = delta * p.scale;

  f32x16 dqacc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < 16; ++j) dqacc[mb][j] = 0.f;

  Streamed<T, DP, DMA> k_rows, v_rows;
  k_rows.init(kb, p.ks[2], tid);
  v_rows.init(vb, p.vs[2], tid);
  auto fetch = [&](int kc0, int buffer) {
    k_rows.fetch(kc0, kv_end, p.d, smem + buffer * BUF_BYTES, tid);
    v_rows.fetch(kc0, kv_end, p.d, smem + buffer * BUF_BYTES + TILE_BYTES, tid);
  };
  const uint32_t row_off = streamed_row_offset<DP>(l32, hh);
  const uint32_t col_off = streamed_column_offset<DP>(lane);
  // bit mode: the lane's query row of the mask, two words (64 keys) per chunk, requested one chunk ahead of their use
  [[maybe_unused]] uint32_t chunk_words[kChunk / 32] = {}, next_words[kChunk / 32] = {};
  auto fetch_words = [&](int kc0, uint32_t (&dst)[kChunk / 32]) {
    const int wpr = (p.Tk + 31) / 32;
    const uint32_t* row = p.bit_words + b * p.bits_bs + static_cast<int64_t>(qi < p.Tq ? qi : 0) * wpr;
    const uint32_t* valid = p.key_valid != nullptr ? reinterpret_cast<const uint32_t*>(p.key_valid) + static_cast<int64_t>(b) * wpr : nullptr;
#pragma unroll
    for (int t = 0; t < kChunk / 32; ++t) {
      const int w = kc0 / 32 + t;
      const bool inside = qi < p.Tq && w < wpr;  // a tile at or beyond Tk has no word
      dst[t] = inside ? row[w] : 0u;
      if (inside && valid != nullptr) dst[t] &= valid[w];
    }
  };
  if (BITS && kv_end > 0) fetch_words(0, chunk_words);
  if (kv_end > 0) fetch(0, 0);
  int buf = 0;
  for (int kc0 = 0; kc0 < kv_end; kc0 += kChunk) {
    if (BITS && !DMA && kc0 + kChunk < kv_end) fetch_words(kc0 + kChunk, next_words);
    if (DMA) {
      vm_wait<0>();     // this wavefront's pieces of the chunk have landed ...
      __syncthreads();  // ... everyone's have, and everyone is done reading the other buffer
      if (BITS && kc0 + kChunk < kv_end) fetch_words(kc0 + kChunk, next_words);  // (in front of the wait it would be waited for)
      if (kc0 + kChunk < kv_end) fetch(kc0 + kChunk, buf ^ 1);
    } else {
      if (kc0 > 0) __syncthreads();  // every wavefront is done reading the previous chunk
      k_rows.commit(smem, tid);
      v_rows.commit(smem + TILE_BYTES, tid);
      __syncthreads();
      if (kc0 + kChunk < kv_end) fetch(kc0 + kChunk, 0);
    }
    const uint8_t* kt_rows = smem + buf * BUF_BYTES;
    const uint32_t col_addr = lds_offset(kt_rows) + col_off;
    if (DMA) buf ^= 1;
    static_for<kChunk / 32>([&](auto kt_tag) {
      constexpr int kt = decltype(kt_tag)::value;
      if (kc0 + kt * 32 >= kv_end || !wave_active) return;  // wavefront-uniform
      if (p.causal && kc0 + kt * 32 > q_begin + wave * 32 + 31) return;  // every key of the tile lies after the queries
      f32x16 sacc, dpacc;
#pragma unroll
      for (int j = 0; j < 16; ++j) sacc[j] = dpacc[j] = 0.f;
      vec_t ka[KSTEPS], va[KSTEPS];
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        const uint32_t off = kt * 32 * ROWB + (row_off ^ (s * 32));
        ka[s] = *reinterpret_cast<const vec_t*>(kt_rows + off);
        va[s] = *reinterpret_cast<const vec_t*>(kt_rows + TILE_BYTES + off);
      }
      [[maybe_unused]] vec4_t columns[2][2];
      if (kAhead) {  // requested together and in front of their use (see attn_bwd_fused_kernel)
        fetch_columns<T, DP>(columns, col_addr + kt * 32 * ROWB);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        sacc = Mfma32<T>::run(ka[s], qf[s], sacc);
        dpacc = Mfma32<T>::run(va[s], dof[s], dpacc);
      }
      // only a tile that crosses the end of the keys or the causal diagonal needs per-element tests
      const int k_tile = kc0 + kt * 32;
      const bool tail = k_tile + 32 > kv_end || (p.causal && k_tile + 31 > q_begin + wave * 32);
      if (tail) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int key = k_tile + (j / 4) * 8 + hh * 4 + (j % 4);
          if (key >= kv_end || (p.causal && key > qi)) sacc[j] = -INFINITY;
        }
      }
      vec_t dsb[2];
      if (MODE == kMaskBits) {
        const uint32_t word = chunk_words[kt] >> (hh * 4);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float prob = where_bit(__builtin_amdgcn_exp2f(fmaf(sacc[j], c, -lse2)), word, (j / 4) * 8 + (j % 4), 1);
          dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dpacc[j], p.scale, -delta_scaled));
        }
      } else if (MODE == kMaskBitsDropout) {
        const uint32_t word = chunk_words[kt];
        const bool aligned = (p.Tk % 4 == 0) && (reinterpret_cast<uintptr_t>(p.drop_mask) % 4 == 0) &&
                             p.mask_bs % 4 == 0 && p.mask_hs % 4 == 0;
        const uint8_t* row = p.drop_mask + b * p.mask_bs + h * p.mask_hs + static_cast<int64_t>(qi < p.Tq ? qi : 0) * p.Tk;
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
          const uint32_t keep = qi < p.Tq ? keep_bytes4(row, k_tile + jq * 8 + hh * 4, p.Tk, aligned) : 0u;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = jq * 4 + e;
            const bool visible = ((word >> (jq * 8 + hh * 4 + e)) & 1u) != 0u;
            const float prob = visible ? __builtin_amdgcn_exp2f(fmaf(sacc[j], c, -lse2)) : 0.f;
            const float dp = ((keep >> (8 * e)) & 0xffu) != 0u ? dpacc[j] * p.drop_scale : 0.f;
            dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dp, p.scale, -delta_scaled));
          }
        }
      } else if (MODE != kMaskNone) {
        const bool aligned = (p.Tk % 4 == 0) && (reinterpret_cast<uintptr_t>(p.drop_mask) % 4 == 0) &&
                             p.mask_bs % 4 == 0 && p.mask_hs % 4 == 0;
        const uint8_t* row = p.drop_mask + b * p.mask_bs + h * p.mask_hs + static_cast<int64_t>(qi < p.Tq ? qi : 0) * p.Tk;
        const bool with_valid = MODE == kMaskVisible && p.key_valid != nullptr;  // uniform
        const uint8_t* valid_row = with_valid ? p.key_valid + static_cast<int64_t>(b) * p.Tk : nullptr;
        const bool valid_aligned = with_valid && (p.Tk % 4 == 0) && (reinterpret_cast<uintptr_t>(p.key_valid) % 4 == 0);
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
          const uint32_t keep = qi < p.Tq ? keep_bytes4(row, k_tile + jq * 8 + hh * 4, p.Tk, aligned) : 0u;
          const uint32_t kval = with_valid ? keep_bytes4(valid_row, k_tile + jq * 8 + hh * 4, p.Tk, valid_aligned) : ~0u;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = jq * 4 + e;
            const bool on = ((keep >> (8 * e)) & 0xffu) != 0u && ((kval >> (8 * e)) & 0xffu) != 0u;
            float prob = __builtin_amdgcn_exp2f(fmaf(sacc[j], c, -lse2));
            if (DROPOUT) {
              const float dp = on ? dpacc[j] * p.drop_scale : 0.f;
              dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dp, p.scale, -delta_scaled));
            } else {
              prob = on ? prob : 0.f;
              dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dpacc[j], p.scale, -delta_scaled));
            }
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float prob = __builtin_amdgcn_exp2f(fmaf(sacc[j], c, -lse2));
          dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dpacc[j], p.scale, -delta_scaled));
        }
      }
      if constexpr (kAhead) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) dqacc[0] = Mfma32<T>::run(join(columns[s2][0], columns[s2][1]), dsb[s2], dqacc[0]);
      } else {
        accumulate_columns<T, DP, kt * 32 * ROWB>(dqacc, dsb, col_addr);
      }
    });
    if (BITS) {
#pragma unroll
      for (int t = 0; t < kChunk / 32; ++t) chunk_words[t] = next_words[t];
    }
  }
  __syncthreads();  // the staging buffers now hold the output tiles
  store_owned<T, DP>(dqacc, smem + wave * (32 * OROW), dqb, p.dqs[2], q_begin + wave * 32, COMPACT ? len : p.Tq, p.d, lane);
}

template <typename T, int DP, bool DMA, int MODE = kMaskNone, bool COMPACT = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu((DP == 32 ? 4 : 3) - (DMA ? 0 : 1)))) void attn_bwd_dkv_kernel(const AttnBwdParams p) {
  constexpr bool DROPOUT = MODE == kMaskDropout || MODE == kMaskBitsDropout;
  constexpr bool BITS = MODE == kMaskBits || MODE == kMaskBitsDropout;
  typedef typename Vec8<T>::type vec_t;
  constexpr int KSTEPS = DP / 16, MB = DP / 32;
  constexpr int ROWB = DP * 2, TILE_BYTES = kChunk * ROWB;
  // a chunk of Q, of dO, then its row statistics; bit mode: then the mask words of the chunk's rows for the 32 keys of
  // each wavefront, [wavefront][row]
  constexpr int kWaves = kThreads / kWave;
  static_assert(kThreads == kWaves * kChunk, "one mask word per thread and chunk");
  constexpr int BUF_BYTES = 2 * TILE_BYTES + 2 * kChunk * 4 + (BITS ? kWaves * kChunk * 4 : 0);
  constexpr int NBUF = DMA ? 2 : 1;
  constexpr int OROW = DP * 2 + 16;
  constexpr int OUT_BYTES = (kThreads / kWave) * 32 * OROW;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NBUF * BUF_BYTES > OUT_BYTES ? NBUF * BUF_BYTES : OUT_BYTES];

  const uint32_t logical = xcd_remap(blockIdx.x, p.total);
  const int blk = static_cast<int>(logical % p.nblk);
  const int bh = static_cast<int>(logical / p.nblk);
  const int h = bh % p.H, b = bh / p.H;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, l32 = lane % 32, hh = lane / 32;
  const T* qb = head_rows<COMPACT>(static_cast<const T*>(p.q), p.qs, p, b, h);
  const T* kb = head_rows<COMPACT>(static_cast<const T*>(p.k), p.ks, p, b, h);
  const T* vb = head_rows<COMPACT>(static_cast<const T*>(p.v), p.vs, p, b, h);
  const T* dob = head_rows<COMPACT>(static_cast<const T*>(p.dout), p.dos, p, b, h);
  T* dkb = head_rows<COMPACT>(static_cast<T*>(p.dk), p.dks, p, b, h);
  T* dvb = head_rows<COMPACT>(static_cast<T*>(p.dv), p.dvs, p, b, h);

  int len = p.Tk;
  if (p.key_lengths != nullptr) {
    len = p.key_lengths[b];
    len = len < 0 ? 0 : (len > p.Tk ? p.Tk : len);
  }
  const int q_valid = p.zero_pad ? (len < p.Tq ? len : p.Tq) : p.Tq;
  const int k_begin = blk * kOwn;
  const int kj = k_begin + wave * 32 + l32;
  // visibility mode: whether the lane's key can be seen at all (its own byte of the key validity, if one was given)
  // bit mode: column (kj / 32) of the sample's word matrix; (k_begin + wave * 32) is a multiple of 32, so the wavefront's
  // keys share the word and key kj is bit l32
  [[maybe_unused]] const int bit_wpr = (p.Tk + 31) / 32;
  [[maybe_unused]] bool key_seen = kj < p.Tk;
  if (MODE == kMaskVisible && key_seen && p.key_valid != nullptr) key_seen = p.key_valid[static_cast<int64_t>(b) * p.Tk + kj] != 0;
  if (BITS && key_seen && p.key_valid != nullptr)
    key_seen = ((reinterpret_cast<const uint32_t*>(p.key_valid)[static_cast<int64_t>(b) * ((p.Tk + 31) / 32) + kj / 32] >> (kj % 32)) & 1u) != 0u;
  [[maybe_unused]] const int key_bits = key_seen ? 1 : 0;  // (a field of no bits is zero: nothing sees the key)
  const bool k_ok = kj < len;
  // queries that can see a key of this block: all valid ones, or (causal) those at or after the block's first key
  const int q_start = p.causal ? (k_begin / kChunk) * kChunk : 0;

  vec_t kf[KSTEPS], vf[KSTEPS];
  load_owned<T, DP>(kb, p.ks[2], kj, k_ok, p.d, hh, kf);
  load_owned<T, DP>(vb, p.vs[2], kj, k_ok, p.d, hh, vf);
  f32x16 dkacc[MB], dvacc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < 16; ++j) dkacc[mb][j] = dvacc[mb][j] = 0.f;
  const float c = p.scale * 1.4426950408889634f;
  // With mask bits the products dP start from -D: four registers less at their peak, without which the kernel spills (d = 32, masked
  // blocks of 128 x 403 tokens 87 -> 71 us). Without them the statistics' way into the accumulators only delays the first product
  // (1024 x 512 tokens 490 -> 512 us). The 1 / sqrt(d) of dS then multiplies dK at the end; in fp16, whose range the unscaled dS
  // could leave, it multiplies every element.
  constexpr bool START_D = MODE == kMaskBits;
  constexpr bool LATE_SCALE = START_D && std::is_same<T, bf16_t>::value;
  const int64_t stat0 = (static_cast<int64_t>(b) * p.H + h) * p.Tq;

  if (k_begin < len) {  // workgroup-uniform: a block of padding keys gets zero gradients without any work
    Streamed<T, DP, DMA> q_rows, do_rows;
    q_rows.init(qb, p.qs[2], tid);
    do_rows.init(dob, p.dos[2], tid);
    float lse_next = -INFINITY, delta_next = 0.f;
    [[maybe_unused]] uint32_t word_next = 0u;
    auto fetch = [&](int qc0, int buffer) {
      q_rows.fetch(qc0, q_valid, p.d, smem + buffer * BUF_BYTES, tid);
      do_rows.fetch(qc0, q_valid, p.d, smem + buffer * BUF_BYTES + TILE_BYTES, tid);
      if (tid < kChunk) {
        const int qi = qc0 + tid;
        lse_next = qi < q_valid ? p.lse[stat0 + qi] : -INFINITY;
        delta_next = qi < q_valid ? p.delta[stat0 + qi] : 0.f;
      }
      if (BITS) {  // thread (w, r): the word of query row qc0 + r that covers the keys of wavefront w
        const int qi = qc0 + tid % kChunk, key0 = k_begin + (tid / kChunk) * 32;
        word_next = (qi < q_valid && key0 < p.Tk) ? p.bit_words[b * p.bits_bs + static_cast<int64_t>(qi) * bit_wpr + key0 / 32] : 0u;
      }
    };
    // the row statistics travel through registers: base-2 log-sum-exp (+inf: the row carries nothing, exp2(x - inf) = 0)
    // and -D_i, times 1 / sqrt(d) where that is not left to the end
    auto commit_stats = [&](int buffer) {
      if (tid < kChunk) {
        float* stats = reinterpret_cast<float*>(smem + buffer * BUF_BYTES + 2 * TILE_BYTES);
        stats[tid] = lse_next > -INFINITY ? lse_next * 1.4426950408889634f : INFINITY;
        stats[kChunk + tid] = START_D ? -delta_next : -delta_next * p.scale;
      }
      if (BITS)
        reinterpret_cast<uint32_t*>(smem + buffer * BUF_BYTES + 2 * TILE_BYTES + 2 * kChunk * 4)[tid] = word_next;
    };
    const uint32_t row_off = streamed_row_offset<DP>(l32, hh);
    const uint32_t col_off = streamed_column_offset<DP>(lane);
    if (q_start < q_valid) {
      fetch(q_start, 0);
      if (DMA) commit_stats(0);
    }
    int buf = 0;
    for (int qc0 = q_start; qc0 < q_valid; qc0 += kChunk) {
      const bool more = qc0 + kChunk < q_valid;
      if (DMA) {
        vm_wait<0>();     // this wavefront's pieces of the chunk have landed ...
        __syncthreads();  // ... everyone's have (and the statistics), and everyone is done reading the other buffer
        if (more) fetch(qc0 + kChunk, buf ^ 1);
      } else {
        if (qc0 > q_start) __syncthreads();  // every wavefront is done reading the previous chunk
        q_rows.commit(smem, tid);
        do_rows.commit(smem + TILE_BYTES, tid);
        commit_stats(0);
        __syncthreads();
        if (more) fetch(qc0 + kChunk, 0);
      }
      const uint8_t* q_tile = smem + buf * BUF_BYTES;
      const float* sLse = reinterpret_cast<const float*>(q_tile + 2 * TILE_BYTES);
      const float* sDelta = sLse + kChunk;
      [[maybe_unused]] const uint32_t* sWords = reinterpret_cast<const uint32_t*>(sDelta + kChunk) + wave * kChunk;
      const uint32_t q_col_addr = lds_offset(q_tile) + col_off;
      if (DMA) buf ^= 1;
      static_for<kChunk / 32>([&](auto qt_tag) {
        constexpr int qt = decltype(qt_tag)::value;
        if (qc0 + qt * 32 >= q_valid || k_begin + wave * 32 >= len) return;  // wavefront-uniform
        if (p.causal && qc0 + qt * 32 + 31 < k_begin + wave * 32) return;     // every query of the tile lies before the keys
        f32x16 sacc, dpacc;
#pragma unroll
        for (int j = 0; j < 16; ++j) sacc[j] = dpacc[j] = 0.f;
        if (START_D) {
#pragma unroll
          for (int jq = 0; jq < 4; ++jq) {
            const f32x4 d4 = *reinterpret_cast<const f32x4*>(&sDelta[qt * 32 + jq * 8 + hh * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) dpacc[jq * 4 + e] = d4[e];
          }
        }
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
          const uint32_t off = qt * 32 * ROWB + (row_off ^ (s * 32));
          const vec_t qa = *reinterpret_cast<const vec_t*>(q_tile + off);
          const vec_t da = *reinterpret_cast<const vec_t*>(q_tile + TILE_BYTES + off);
          sacc = Mfma32<T>::run(qa, kf[s], sacc);
          dpacc = Mfma32<T>::run(da, vf[s], dpacc);
        }
        // (causal) a query before the key: the score becomes -inf, the probability 0; only a tile that crosses the
        // causal diagonal needs per-element tests. A padded key of the lane (zeros in kf and vf) collects finite
        // values in its own accumulator column only, which is cleared after the loop.
        const bool diagonal = p.causal && qc0 + qt * 32 < k_begin + wave * 32 + 31;
        if (diagonal) {  // wavefront-uniform: the other tiles pay nothing for the triangle
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (kj > qc0 + qt * 32 + (j / 4) * 8 + hh * 4 + (j % 4)) sacc[j] = -INFINITY;
        }
        vec_t pb[2], dsb[2];
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
          const int r0 = qt * 32 + jq * 8 + hh * 4;  // four consecutive queries of the chunk
          const f32x4 l4 = *reinterpret_cast<const f32x4*>(&sLse[r0]);
          [[maybe_unused]] f32x4 d4 = {0.f, 0.f, 0.f, 0.f};
          if (!START_D) d4 = *reinterpret_cast<const f32x4*>(&sDelta[r0]);
          [[maybe_unused]] u32x4 w4 = {0u, 0u, 0u, 0u};
          if (BITS) w4 = *reinterpret_cast<const u32x4*>(&sWords[r0]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = jq * 4 + e;
            float prob = __builtin_amdgcn_exp2f(fmaf(sacc[j], c, -l4[e]));
            if (MODE == kMaskBits) {
              // the lane owns key kj; register j is query qc0 + r0 + e: bit l32 of that row's word for the wavefront's keys
              prob = where_bit(prob, w4[e], l32, key_bits);
              pb[j / 8][j % 8] = static_cast<T>(prob);
              dsb[j / 8][j % 8] = static_cast<T>(prob * (LATE_SCALE ? dpacc[j] : dpacc[j] * p.scale));
            } else if (MODE == kMaskBitsDropout) {
              const int qrow = qc0 + r0 + e;
              prob = (key_seen && ((w4[e] >> l32) & 1u) != 0u) ? prob : 0.f;
              const bool keep = qrow < p.Tq && kj < p.Tk &&
                                p.drop_mask[b * p.mask_bs + h * p.mask_hs + static_cast<int64_t>(qrow) * p.Tk + kj] != 0;
              pb[j / 8][j % 8] = static_cast<T>(keep ? prob * p.drop_scale : 0.f);
              dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(keep ? dpacc[j] * p.drop_scale : 0.f, p.scale, d4[e]));
            } else if (MODE != kMaskNone) {
              // the lane owns key kj; register j is query qc0 + r0 + e: one mask byte per register
              const int qrow = qc0 + r0 + e;
              const bool keep = qrow < p.Tq && key_seen &&
                                p.drop_mask[b * p.mask_bs + h * p.mask_hs + static_cast<int64_t>(qrow) * p.Tk + kj] != 0;
              if (DROPOUT) {
                pb[j / 8][j % 8] = static_cast<T>(keep ? prob * p.drop_scale : 0.f);
                dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(keep ? dpacc[j] * p.drop_scale : 0.f, p.scale, d4[e]));
              } else {
                prob = keep ? prob : 0.f;
                pb[j / 8][j % 8] = static_cast<T>(prob);
                dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dpacc[j], p.scale, d4[e]));
              }
            } else {
              pb[j / 8][j % 8] = static_cast<T>(prob);
              dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dpacc[j], p.scale, d4[e]));
            }
          }
        }
        accumulate_columns2<T, DP, qt * 32 * ROWB>(dvacc, pb, q_col_addr + TILE_BYTES, dkacc, dsb, q_col_addr);
      });
      if (DMA && more) commit_stats(buf);  // the next chunk's statistics: the barrier above publishes them
    }
  }
  if (LATE_SCALE) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) dkacc[mb][j] *= p.scale;
  }
  if (!k_ok) {  // a key in the padding receives no gradient
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) dkacc[mb][j] = dvacc[mb][j] = 0.f;
  }
  __syncthreads();
  uint8_t* tile = smem + wave * (32 * OROW);
  const int k_store_end = COMPACT ? len : p.Tk;
  store_owned<T, DP>(dkacc, tile, dkb, p.dks[2], k_begin + wave * 32, k_store_end, p.d, lane);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  store_owned<T, DP>(dvacc, tile, dvb, p.dvs[2], k_begin + wave * 32, k_store_end, p.d, lane);
}

template <typename T>
struct Mfma16;
template <>
struct Mfma16<bf16_t> {
  static __device__ __forceinline__ f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16<f16_t> {
  static __device__ __forceinline__ f32x4 run(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// dQ, dK and dV of one (batch, head) in one workgroup, for samples whose keys it can hold: S, dP and the exponentials are
// formed once instead of twice (five products per pair of tiles instead of seven) and every tensor is read once.
// Wavefront w owns the 32-key tiles w, w + 4, ... (NT of them: their dK / dV accumulators and V fragments stay in
// registers, NT * DP = 64 or 128), K lies in LDS as a whole, the queries stream through LDS in chunks of 32 rows. A lane
// owns a key, so P and dS come out of the first products as the B operands of dV and dK; dQ contracts over the keys
// instead: the dS tiles of all wavefronts meet in LDS ([key][query], 16 bits as every operand) and each wavefront forms
// its own 16 queries x 16 features (DP = 64: twice) of dQ over all key tiles, so dQ, too, has one writer per element and
// a fixed order. Every sum is formed in the order of the two kernels and every value rounded as there, so that the
// gradients are theirs to the bit, whichever route a batch's size takes. (Without a mask, D added up over eight lanes a row, the start
// value of dP, and 1 / sqrt(d) at the end save three instructions per pair, 1024 x 8 x 512 x 32 604 instead of 638 us, 2048 x 4 x 256 x 64
// 371 instead of 383, but move a quarter of dQ and dK at d = 32 by a rounding, which a few layers make 0.2 % of every gradient.)
// Under mask bits the two kernels round the dS of dQ and that of dK differently (START_D there), so that dP is formed twice, one behind the
// other. Two wavefronts a SIMD instead of three leave the registers for it: with three, 16 to 36 of them are spilled (256 rows, 8192 pairs
// of 32 features 340 instead of 290 us; 64 rows of 64 features 192 instead of 123). One dP and the scale at the end moved dK, at d = 64 dQ,
// by roundings: 312 and 133 us there, with three wavefronts.
// A pair of tiles is some 490 cycles of vector instructions and 320 of products, but also a chain from LDS reads to products to exponentials to
// products, which two or three wavefronts a SIMD do not cover. Left alone, the compiler puts each read in front of the instruction that takes
// it: nine memory latencies per pair. With 32 features the operands, the rows' values and the columns of the second products are therefore
// requested behind scheduling fences ahead of their use, and dQ's contraction requests the next two tiles in front of the products of two (as
// nested branches: one behind the other they hold both groups' registers across all of them, and spill). 64 features leave the registers for
// the rows' values alone, and without mask bits. K's and dS's pieces lie so that a transposed read has no two lanes on one bank (both had two, a
// quarter of the LDS cycles). 1024 x 8 x 512 x 32, lengths ~ U{64..512} 718 -> 670 us, all 512 1215 -> 1115, causal (600 samples) 297 -> 272;
// 1024 x 8 x 256 x 32 203 -> 191; 2048 x 4 x 256 x 64 369 -> 353; 110 rows of 64 151 -> 146.
template <int DP, int NT, bool BITS>
struct FusedLayout {
  static constexpr int kRows = 32;                                     // streamed queries per step
  static constexpr int ROWB = DP * 2, TILE_BYTES = kRows * ROWB;
  static constexpr int kWaves = kThreads / kWave, kTiles = kWaves * NT;  // key tiles of 32 rows
  static constexpr int K_BYTES = kTiles * TILE_BYTES, DS_BYTES = kTiles * kRows * 64;
  static constexpr int WORD_BYTES = BITS ? kTiles * kRows * 4 : 0;      // [tile][row]
  static constexpr int BUF_BYTES = 2 * TILE_BYTES + WORD_BYTES;         // Q, dO, words
  static constexpr int STAT_BYTES = (BITS ? 3 : 2) * kTiles * kRows * 4;  // log-sum-exp and -D / sqrt(d) of every query; -D
  static constexpr int BYTES = K_BYTES + DS_BYTES + 2 * BUF_BYTES + STAT_BYTES;
  static constexpr int kWavesPerSimd = NT * DP == 128 || BITS ? 2 : 3;
  // What a pair of tiles reads from LDS is requested ahead of its use, as far as the registers go (see the loop over the tiles).
  static constexpr bool kOperandsAhead = DP == 32;
  static constexpr bool kRowsAhead = DP == 32 || (NT == 2 && !BITS);
};

template <typename T, int DP, int NT, int MODE, bool COMPACT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(FusedLayout<DP, NT, MODE == kMaskBits>::kWavesPerSimd,
                                                                          FusedLayout<DP, NT, MODE == kMaskBits>::kWavesPerSimd)))
void attn_bwd_fused_kernel(const AttnBwdParams p) {
  constexpr bool BITS = MODE == kMaskBits;
  static_assert(MODE == kMaskNone || BITS, "the other masks are read per element by the two kernels above");
  typedef typename Vec8<T>::type vec_t;
  typedef typename Vec8<T>::half_type vec4_t;
  typedef FusedLayout<DP, NT, BITS> L;
  constexpr int KSTEPS = DP / 16, MB = DP / 32, C8 = DP / 8, kRows = L::kRows, ROWB = L::ROWB, TILE_BYTES = L::TILE_BYTES;
  constexpr int kWaves = L::kWaves;
  [[maybe_unused]] constexpr int kWords = L::kTiles * kRows;
  constexpr bool LATE_SCALE = BITS && std::is_same<T, bf16_t>::value;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[L::BYTES];
  uint8_t* const k_image = smem;
  uint8_t* const ds_image = smem + L::K_BYTES;
  uint8_t* const buffers = smem + L::K_BYTES + L::DS_BYTES;

  const int bh = static_cast<int>(xcd_remap(blockIdx.x, p.total));
  const int h = bh % p.H, b = bh / p.H;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, l32 = lane % 32, hh = lane / 32;
  const T* qb = head_rows<COMPACT>(static_cast<const T*>(p.q), p.qs, p, b, h);
  const T* kb = head_rows<COMPACT>(static_cast<const T*>(p.k), p.ks, p, b, h);
  const T* vb = head_rows<COMPACT>(static_cast<const T*>(p.v), p.vs, p, b, h);
  const T* ob = head_rows<COMPACT>(static_cast<const T*>(p.o), p.os, p, b, h);
  const T* dob = head_rows<COMPACT>(static_cast<const T*>(p.dout), p.dos, p, b, h);
  T* dqb = head_rows<COMPACT>(static_cast<T*>(p.dq), p.dqs, p, b, h);
  T* dkb = head_rows<COMPACT>(static_cast<T*>(p.dk), p.dks, p, b, h);
  T* dvb = head_rows<COMPACT>(static_cast<T*>(p.dv), p.dvs, p, b, h);

  int len = p.Tk;
  if (p.key_lengths != nullptr) {
    len = p.key_lengths[b];
    len = len < 0 ? 0 : (len > p.Tk ? p.Tk : len);
  }
  const int q_valid = p.zero_pad ? (len < p.Tq ? len : p.Tq) : p.Tq;
  // The wavefront's key tiles are own, own + 4, ...: with a number of tiles that 4 does not divide the wavefronts with one tile more
  // lie on other SIMDs in other workgroups.
  const int own = __builtin_amdgcn_readfirstlane((wave + bh + bh / 32) % (kThreads / kWave));
  const int n_tiles = (len + 31) / 32;           // at most L::kTiles: the host checks Tk
  const int q_end = n_tiles > 0 ? q_valid : 0;   // rows of dQ at or beyond it are zero
  const float c = p.scale * 1.4426950408889634f;
  const int64_t stat0 = (static_cast<int64_t>(b) * p.H + h) * p.Tq;
  [[maybe_unused]] const int wpr = (p.Tk + 31) / 32;

  f32x16 dkacc[NT][MB], dvacc[NT][MB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) dkacc[t][mb][j] = dvacc[t][mb][j] = 0.f;

  if (q_end > 0) {
    // ---- a chunk of Q and dO: 1 KB transfers straight into LDS, dealt to the wavefronts; rows at or beyond q_valid
    // repeat the last valid one (their probabilities are zeros). Row r of a tile: 16-byte piece x lies at x ^ row_swizzle(r).
    auto transfer = [&](const T* base, int64_t stride, int row0, int row_end, int slot, uint8_t* tile) {
      const int r = slot * (kWave / C8) + lane / C8;
      const int piece = (lane % C8) ^ row_swizzle<DP>(r);
      int row = row0 + r;
      row = row < row_end ? row : row_end - 1;
      lds_dma16_offset(base, __umul24(static_cast<uint32_t>(row), static_cast<uint32_t>(stride) * 2u) + static_cast<uint32_t>(piece * 16),
                       tile + slot * 1024);
    };
    constexpr int kSlots = TILE_BYTES / 1024;  // per operand of a chunk: 2 or 4
    auto fetch_chunk = [&](int qc0, uint8_t* buf) {
#pragma unroll
      for (int i = 0; i < 2 * kSlots / kWaves; ++i) {
        const int slot = wave + i * kWaves;  // wavefront-uniform
        if (slot < kSlots)
          transfer(qb, p.qs[2], qc0, q_valid, slot, buf);
        else
          transfer(dob, p.dos[2], qc0, q_valid, slot - kSlots, buf + TILE_BYTES);
      }
    };
    // words of the chunk's rows for every key tile, [tile][row], one per lane and transfer; rows and tiles that do not exist repeat
    // the last one (their probabilities are zeros, or nobody reads them)
    auto fetch_words = [&](int qc0, uint8_t* buf) {
#pragma unroll
      for (int i = 0; i < (kWords + kThreads - 1) / kThreads; ++i) {
        const int slot0 = i * kThreads + wave * kWave;
        if (slot0 < kWords) {  // wavefront-uniform
          const int slot = slot0 + lane;
          int tile = slot / kRows, qi = qc0 + slot % kRows;
          tile = tile < n_tiles ? tile : n_tiles - 1;
          qi = qi < q_valid ? qi : q_valid - 1;
          lds_dma4(p.bit_words + b * p.bits_bs + static_cast<int64_t>(qi) * wpr + tile, buf + 2 * TILE_BYTES + slot0 * 4);
        }
      }
    };
    // The statistics of all queries: base-2 log-sum-exp, +inf for a row that carries nothing: exp2(x - inf) = 0, and -D / sqrt(d) (with
    // mask bits -D, too), two threads a row. Rows of the last chunk at or beyond q_valid among them.
    float* const stats = reinterpret_cast<float*>(buffers + 2 * L::BUF_BYTES);
    constexpr int kStatRows = kThreads / 2, kStatUnroll = 2;  // rows per pass, passes in flight
    auto row_stats = [&](int row0) {
      const int half = tid % 2;
      vec_t of[kStatUnroll][KSTEPS], dof[kStatUnroll][KSTEPS];
      float lse[kStatUnroll];
#pragma unroll
      for (int u = 0; u < kStatUnroll; ++u) {
        const int row = row0 + u * kStatRows + tid / 2;
        lse[u] = row < q_valid ? p.lse[stat0 + row] : -INFINITY;
        load_owned<T, DP>(ob, p.os[2], row, row < q_valid, p.d, half, of[u]);
        load_owned<T, DP>(dob, p.dos[2], row, row < q_valid, p.d, half, dof[u]);
      }
#pragma unroll
      for (int u = 0; u < kStatUnroll; ++u) {
        const int row = row0 + u * kStatRows + tid / 2;
        if (row0 + u * kStatRows >= q_valid) break;  // uniform
        float delta = 0.f;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
          for (int e = 0; e < 8; ++e) delta = fmaf(static_cast<float>(of[u][s][e]), static_cast<float>(dof[u][s][e]), delta);
        delta = group_sum<2>(delta);
        if (half == 0 && row < L::kTiles * kRows) {
          stats[row] = lse[u] > -INFINITY ? lse[u] * 1.4426950408889634f : INFINITY;
          stats[L::kTiles * kRows + row] = -delta * p.scale;
          if (BITS) stats[2 * L::kTiles * kRows + row] = -delta;
        }
      }
    };

    if (BITS) fetch_words(0, buffers);
    for (int slot = wave; slot < n_tiles * kSlots; slot += kWaves)
      transfer(kb, p.ks[2], 0, len, slot, k_image);
    fetch_chunk(0, buffers);
    vec_t vf[NT][KSTEPS];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int key = (own + t * kWaves) * 32 + l32;
      load_owned<T, DP>(vb, p.vs[2], key, key < len, p.d, hh, vf[t]);
    }
    for (int row0 = 0; row0 < q_valid; row0 += kStatUnroll * kStatRows) row_stats(row0);
    // bit t: the lane's key of the wavefront's tile t is valid as a key
    [[maybe_unused]] uint32_t seen = ~0u;
    if (BITS && p.key_valid != nullptr) {
      seen = 0u;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int tile = own + t * kWaves;
        if (tile < n_tiles)
          seen |= ((reinterpret_cast<const uint32_t*>(p.key_valid)[static_cast<int64_t>(b) * wpr + tile] >> l32) & 1u) << t;
      }
    }

    const uint32_t row_off = streamed_row_offset<DP>(l32, hh);
    const uint32_t col_off = streamed_column_offset<DP>(lane);
    // dS in LDS: rows of 32 queries per key, the 8-byte piece x of key r at x ^ ds_swizzle(r): one piece of 32 keys (a write) and four
    // pieces of eight consecutive keys (half of a transposed read below) cover all 64 banks.
    auto ds_swizzle = [](int r) { return ((r >> 3) & 3) | (r & 4); };
    const uint32_t ds_write = static_cast<uint32_t>(l32 * 64);
    const int g16 = lane / 16, i16 = lane % 16, q_half = wave % 2, d_col = wave / 2;
    uint32_t ds_read[2], k_read[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // of the tile: one transposed read holds four keys, in the order in which accumulate_columns has them (the matrix unit adds a
      // product's terms in theirs)
      const int key = 16 * (g16 / 2) + 4 * (g16 % 2) + 8 * half + i16 / 4;
      const int piece = 4 * q_half + i16 % 4;        // four queries
      ds_read[half] = lds_offset(ds_image) + static_cast<uint32_t>(key * 64 + ((piece ^ ds_swizzle(key)) * 8));
      const int piece16 = 2 * d_col + (i16 % 4) / 2;  // eight features
      k_read[half] = lds_offset(k_image) + static_cast<uint32_t>(key * ROWB + ((piece16 ^ row_swizzle<DP>(key)) * 16) + (i16 % 2) * 8);
    }

    vm_wait<0>();
    int buf = 0;
    for (int qc0 = 0; qc0 < q_valid; qc0 += kRows) {
      const bool more = qc0 + kRows < q_valid;
      const int q_tile = qc0 / kRows;
      const int tiles = p.causal ? (n_tiles < q_tile + 1 ? n_tiles : q_tile + 1) : n_tiles;  // key tiles these queries see
      uint8_t* const chunk = buffers + buf * L::BUF_BYTES;
      uint8_t* const next = buffers + (buf ^ 1) * L::BUF_BYTES;
      __syncthreads();  // the chunk and its statistics have landed (every wavefront awaited its own transfers); dS is free
      if (more) {
        if (BITS) fetch_words(qc0 + kRows, next);
        fetch_chunk(qc0 + kRows, next);
      }
      const float* s_lse = stats + qc0;
      const float* s_delta = s_lse + L::kTiles * kRows;
      [[maybe_unused]] const uint32_t* s_words = reinterpret_cast<const uint32_t*>(chunk + 2 * TILE_BYTES);
      const uint32_t col_addr = lds_offset(chunk) + col_off;
      static_for<NT>([&](auto t_tag) {
        constexpr int t = decltype(t_tag)::value;
        const int tile = own + t * kWaves;
        if (tile >= tiles) return;  // wavefront-uniform
        f32x16 sacc, dpacc;
#pragma unroll
        for (int j = 0; j < 16; ++j) sacc[j] = dpacc[j] = 0.f;
        vec_t qa[KSTEPS], kf[KSTEPS], da[KSTEPS];
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
          qa[s] = *reinterpret_cast<const vec_t*>(chunk + (row_off ^ (s * 32)));
          kf[s] = *reinterpret_cast<const vec_t*>(k_image + tile * TILE_BYTES + (row_off ^ (s * 32)));
        }
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) da[s] = *reinterpret_cast<const vec_t*>(chunk + TILE_BYTES + (row_off ^ (s * 32)));
        f32x4 l4[2], d4[2];
        [[maybe_unused]] u32x4 w4[2];
        auto row_values = [&](int jq) {  // of the four queries of the accumulators' quarter jq
          l4[jq % 2] = *reinterpret_cast<const f32x4*>(&s_lse[jq * 8 + hh * 4]);
          d4[jq % 2] = *reinterpret_cast<const f32x4*>(&s_delta[jq * 8 + hh * 4]);
          if (BITS) w4[jq % 2] = *reinterpret_cast<const u32x4*>(&s_words[tile * kRows + jq * 8 + hh * 4]);
        };
        if (L::kRowsAhead) row_values(0);
        if (L::kOperandsAhead) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) sacc = Mfma32<T>::run(qa[s], kf[s], sacc);
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) dpacc = Mfma32<T>::run(da[s], vf[t][s], dpacc);
        const int key = tile * 32 + l32;
        // pairs that do not exist get a score of -inf; only the tile at the end of the keys and the one on the causal diagonal test
        if (tile * 32 + 32 > len || (BITS && p.key_valid != nullptr)) {  // wavefront-uniform
          const bool beyond = key >= len || (BITS && ((seen >> t) & 1u) == 0u);
#pragma unroll
          for (int j = 0; j < 16; ++j) sacc[j] = beyond ? -INFINITY : sacc[j];
        }
        if (p.causal && tile == q_tile) {
          const int first = l32 - hh * 4;  // query row (j / 4) * 8 + hh * 4 + j % 4 lies before key l32
#pragma unroll
          for (int j = 0; j < 16; ++j) sacc[j] = first > (j / 4) * 8 + (j % 4) ? -INFINITY : sacc[j];
        }
        vec_t pb[2], dsb[2];
        [[maybe_unused]] vec4_t fd[2][2], fq[2][2];  // columns of dO and Q: the operands of dV and dK
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
          if (!L::kRowsAhead)
            row_values(jq);
          else if (jq < 3)
            row_values(jq + 1);
          if (L::kOperandsAhead && !BITS) {
            if (jq == 2) fetch_columns<T, DP>(fd, col_addr + TILE_BYTES);
            if (jq == 3) fetch_columns<T, DP>(fq, col_addr);
          }
          if (L::kRowsAhead) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = jq * 4 + e;
            float prob = __builtin_amdgcn_exp2f(fmaf(sacc[j], c, -l4[jq % 2][e]));
            if (BITS) prob = where_bit(prob, w4[jq % 2][e], l32, 1);
            pb[j / 8][j % 8] = static_cast<T>(prob);
            dsb[j / 8][j % 8] = static_cast<T>(prob * fmaf(dpacc[j], p.scale, d4[jq % 2][e]));
            if (BITS) sacc[j] = prob;
          }
        }
        uint8_t* const ds_tile = ds_image + tile * (kRows * 64) + ds_write;
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
          vec4_t quad;
#pragma unroll
          for (int e = 0; e < 4; ++e) quad[e] = dsb[jq / 2][(jq % 2) * 4 + e];
          *reinterpret_cast<vec4_t*>(ds_tile + ((2 * jq + hh) ^ ds_swizzle(l32)) * 8) = quad;
        }
        if constexpr (BITS) {  // dK's dS: the products start from -D, 1 / sqrt(d) comes at the end (fp16: before the rounding)
#pragma unroll
          for (int jq = 0; jq < 4; ++jq) {
            const f32x4 d4 = *reinterpret_cast<const f32x4*>(&s_delta[L::kTiles * kRows + jq * 8 + hh * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) dpacc[jq * 4 + e] = d4[e];
          }
#pragma unroll
          for (int s = 0; s < KSTEPS; ++s) {
            const vec_t again = *reinterpret_cast<const vec_t*>(chunk + TILE_BYTES + (row_off ^ (s * 32)));
            dpacc = Mfma32<T>::run(again, vf[t][s], dpacc);
          }
#pragma unroll
          for (int j = 0; j < 16; ++j) dsb[j / 8][j % 8] = static_cast<T>(sacc[j] * (LATE_SCALE ? dpacc[j] : dpacc[j] * p.scale));
        }
        if constexpr (!L::kOperandsAhead) {
          accumulate_columns2<T, DP, 0>(dvacc[t], pb, col_addr + TILE_BYTES, dkacc[t], dsb, col_addr);
        } else {
          if (BITS) {
            fetch_columns<T, DP>(fd, col_addr + TILE_BYTES);
            fetch_columns<T, DP>(fq, col_addr);
          }
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            dvacc[t][0] = Mfma32<T>::run(join(fd[s2][0], fd[s2][1]), pb[s2], dvacc[t][0]);
            dkacc[t][0] = Mfma32<T>::run(join(fq[s2][0], fq[s2][1]), dsb[s2], dkacc[t][0]);
          }
        }
      });
      __syncthreads();  // the dS tiles of every wavefront are in LDS
      f32x4 dqacc[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m) dqacc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      // In groups of key tiles, the next group's operands requested in front of this group's products. What lies beyond the last tile
      // is read (the images have kTiles tiles) but not multiplied.
      constexpr int kGroup = 2 / MB, kGroups = L::kTiles / kGroup;
      vec4_t fs[2][kGroup][2], fk[2][kGroup][MB][2];
      auto fetch_group = [&](auto g_tag) {
        constexpr int g = decltype(g_tag)::value;
#pragma unroll
        for (int i = 0; i < kGroup; ++i) {
          constexpr int first = g * kGroup;
          fs[g % 2][i][0] = read_tr16<T>(ds_read[0] + (first + i) * (kRows * 64));
          fs[g % 2][i][1] = read_tr16<T>(ds_read[1] + (first + i) * (kRows * 64));
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            fk[g % 2][i][m][0] = read_tr16<T>((k_read[0] ^ (m * 64)) + (first + i) * TILE_BYTES);
            fk[g % 2][i][m][1] = read_tr16<T>((k_read[1] ^ (m * 64)) + (first + i) * TILE_BYTES);
          }
        }
      };
      fetch_group(std::integral_constant<int, 0>{});
      auto contract = [&](auto self, auto g_tag) -> void {
        constexpr int g = decltype(g_tag)::value;
        if constexpr (g + 1 < kGroups) fetch_group(std::integral_constant<int, g + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kGroup; ++i)
          if (i == 0 || g * kGroup + i < tiles) {
#pragma unroll
            for (int m = 0; m < MB; ++m)
              dqacc[m] = Mfma16<T>::run(join(fk[g % 2][i][m][0], fk[g % 2][i][m][1]), join(fs[g % 2][i][0], fs[g % 2][i][1]), dqacc[m]);
          }
        if constexpr (g + 1 < kGroups) {
          if ((g + 1) * kGroup < tiles) self(self, std::integral_constant<int, g + 1>{});
        }
      };
      contract(contract, std::integral_constant<int, 0>{});
      vm_wait<0>();  // the next chunk's transfers, before this chunk's stores join the queue
      const int q_row = qc0 + 16 * q_half + i16;
      if (q_row < q_valid) {
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          vec4_t out;
#pragma unroll
          for (int e = 0; e < 4; ++e) out[e] = static_cast<T>(dqacc[m][e]);
          *reinterpret_cast<vec4_t*>(dqb + q_row * p.dqs[2] + 32 * m + 16 * d_col + 4 * g16) = out;
        }
      }
      buf ^= 1;
    }
    __syncthreads();  // the images now hold the output tiles
    uint8_t* out_tile = smem + wave * (32 * (ROWB + 16));
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int key0 = (own + t * kWaves) * 32;
      if (key0 >= n_tiles * 32) break;
      if (LATE_SCALE) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int j = 0; j < 16; ++j) dkacc[t][mb][j] *= p.scale;
      }
      store_owned<T, DP>(dkacc[t], out_tile, dkb, p.dks[2], key0, len, p.d, lane);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      store_owned<T, DP>(dvacc[t], out_tile, dvb, p.dvs[2], key0, len, p.d, lane);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
  if (!COMPACT) {  // rows without a gradient: keys of the padding too, whose sums hold 0 x inf where a gradient is not finite
    vec_t zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = static_cast<T>(0.f);
    const int piece = (tid % C8) * 8;
    for (int row = q_end + tid / C8; row < p.Tq; row += kThreads / C8) *reinterpret_cast<vec_t*>(dqb + row * p.dqs[2] + piece) = zero;
    for (int row = (q_end > 0 ? len : 0) + tid / C8; row < p.Tk; row += kThreads / C8) {
      *reinterpret_cast<vec_t*>(dkb + row * p.dks[2] + piece) = zero;
      *reinterpret_cast<vec_t*>(dvb + row * p.dvs[2] + piece) = zero;
    }
  }
}

bool strides_ok(const int64_t* st) {
  if (!st || st[3] != 1) return false;
  for (int i = 0; i < 3; ++i)
    if (st[i] % 8 != 0 || st[i] < 0) return false;
  return true;
}

// 32-bit source offsets with a 24-bit row multiply: row strides below 4 M elements, sequences below 2^31 bytes.
bool small_offsets(int64_t rows, int64_t stride) {
  return stride < (1 << 22) && rows < (1 << 22) && rows * stride * 2 < (1ll << 31);
}

// The fused kernel where a workgroup can hold a sample's keys (512 of 32 features, 256 of 64) and there are enough (sample, head)
// pairs: it has one workgroup per pair where the two kernels have one per 128 rows. Two kernels / fused in us, lengths ~ U{16..rows}:
//   up to 128 rows (as many workgroups either way):  48 x 32, 256 pairs 9.9 / 9.0, 8192 pairs 65 / 58; 128 x 32, 8192 pairs 126 / 107;
//   128 x 64, 256 pairs 16.9 / 12.8, 16384 pairs 456 / 328.
//   256 x 32:  128 pairs 15.9 / 17.3, 256 pairs 20.1 / 19.1, 512 pairs 27.0 / 24.8, 4096 pairs 156 / 117;  256 x 64:  128 pairs 22.7 / 24.9, 256
//   pairs 30.3 / 27.4, 512 pairs 48 / 39, 8192 pairs 538 / 376. (Between 256 and 512 pairs a few per cent lie on either side.)
//   More rows of 32 features, four key tiles per wavefront and half the wavefronts in flight:  300 rows, 512 pairs 34.6 / 31.0, 1024 pairs
//   55 / 48, 2048 pairs 93 / 82, 8192 pairs 361 / 283;  384 rows, 512 pairs 45.3 / 45.6, 1024 pairs 72 / 66, 2048 pairs 119 / 98;  400 rows, 1024
//   pairs 92 / 71, 8192 pairs 654 / 411;  480 rows, 512 pairs 65 / 67, 1024 pairs 101 / 89;  512 rows, 512 pairs 62 / 61, 1024 pairs 109 / 89, 8192
//   pairs 821 / 589. Causal, 300 rows, 512 pairs 29.8 / 23.4, 512 rows 60 / 45.
// Mask bits: 64 features, 64 rows, 256 pairs 13.5 / 9.5, 8192 pairs 172 / 128, 256 rows, 256 pairs 37 / 36, 512 pairs 57 / 48, 8192 pairs 649 / 472;
// 32 features, 160 rows, 512 pairs 24.0 / 20.0, 256 rows, 512 pairs 31.7 / 29.7, 8192 pairs 345 / 269. Up to 128 rows of 32 features there is
// little to gain, and the second dP loses it where the workgroups are several to a compute unit: 64 rows, 512 pairs 12.2 / 9.9, 1536 pairs
// 22.6 / 21.6, 2048 pairs 25.6 / 27.0, 8192 pairs 76 / 86; 96 rows, 2048 pairs 33.0 / 31.3, 4096 pairs 55.6 / 57.1; 128 rows, 2048 pairs 43.0 /
// 38.5, 3072 pairs 52.6 / 50.7, 6144 pairs 97 / 103. Over 256 rows of 32 features they stay with the two kernels: the words' registers are the
// ones that the four key tiles of a wavefront need (with one dP and before both forms' reads were requested ahead, 300 rows, 1024 pairs 67 / 74,
// 4096 pairs 239 / 274; 403 rows 117 / 116, 436 / 360).
template <typename T, int DP, int MODE, bool COMPACT>
bool launch_bwd_fused(AttnBwdParams p, hipStream_t s) {
  constexpr int kSmall = 64 / DP, kLarge = 128 / DP;  // key tiles per wavefront
  constexpr int kRowsSmall = kSmall * kOwn, kRowsLarge = DP == 32 && MODE == kMaskBits ? kRowsSmall : kLarge * kOwn;
  const int64_t pairs = static_cast<int64_t>(p.B) * p.H;
  const int32_t rows = p.Tq > p.Tk ? p.Tq : p.Tk;
  int64_t enough = rows <= kOwn ? 1 : 512;
  if (DP == 32 && rows > kRowsSmall && !p.causal) enough = 1024;
  if (rows > kRowsLarge || pairs < enough) return false;
  if (DP == 32 && MODE == kMaskBits && rows <= kOwn && pairs > (rows <= 64 ? 1536 : 2048)) return false;
  if (!small_offsets(p.Tq, p.qs[2]) || !small_offsets(p.Tq, p.dos[2]) || !small_offsets(p.Tk, p.ks[2])) return false;
  p.nblk = 1;
  p.total = static_cast<uint32_t>(pairs);
  if (rows <= kRowsSmall)
    hipLaunchKernelGGL((attn_bwd_fused_kernel<T, DP, kSmall, MODE, COMPACT>), dim3(p.total), dim3(kThreads), 0, s, p);
  else if constexpr (kRowsLarge > kRowsSmall)
    hipLaunchKernelGGL((attn_bwd_fused_kernel<T, DP, kLarge, MODE, COMPACT>), dim3(p.total), dim3(kThreads), 0, s, p);
  return true;
}

template <typename T, int DP, int MODE, bool COMPACT>
void launch_bwd_form(AttnBwdParams p, bool register_staging, hipStream_t s) {
  // TAAC_ATTN_REGISTER_STAGING keeps the register-staged kernels for full head dims too (comparison route of the caller).
  const bool direct = p.d == DP && !register_staging;
  if constexpr (MODE == kMaskNone || MODE == kMaskBits) {
    if (direct && launch_bwd_fused<T, DP, MODE, COMPACT>(p, s)) return;
  }
  p.nblk = static_cast<uint32_t>((p.Tq + kOwn - 1) / kOwn);
  p.total = p.nblk * p.B * p.H;
  if (direct && small_offsets(p.Tk, p.ks[2]) && small_offsets(p.Tk, p.vs[2]))
    hipLaunchKernelGGL((attn_bwd_dq_kernel<T, DP, true, MODE, COMPACT>), dim3(p.total), dim3(kThreads), 0, s, p);
  else
    hipLaunchKernelGGL((attn_bwd_dq_kernel<T, DP, false, MODE, COMPACT>), dim3(p.total), dim3(kThreads), 0, s, p);
  p.nblk = static_cast<uint32_t>((p.Tk + kOwn - 1) / kOwn);
  p.total = p.nblk * p.B * p.H;
  if (direct && small_offsets(p.Tq, p.qs[2]) && small_offsets(p.Tq, p.dos[2]))
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<T, DP, true, MODE, COMPACT>), dim3(p.total), dim3(kThreads), 0, s, p);
  else
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<T, DP, false, MODE, COMPACT>), dim3(p.total), dim3(kThreads), 0, s, p);
}

template <typename T, int DP, int MODE>
void launch_bwd_mode(const AttnBwdParams& p, bool register_staging, hipStream_t s) {
  if constexpr (std::is_same<T, bf16_t>::value && (MODE == kMaskNone || MODE == kMaskBits)) {  // what attention_compact_bwd asks for
    if (p.row_offsets != nullptr) return launch_bwd_form<T, DP, MODE, true>(p, register_staging, s);
  }
  launch_bwd_form<T, DP, MODE, false>(p, register_staging, s);
}

template <typename T, int DP>
void launch_bwd_dp(const AttnBwdParams& p, int mode, bool register_staging, hipStream_t s) {
  if (mode == kMaskDropout)
    launch_bwd_mode<T, DP, kMaskDropout>(p, register_staging, s);
  else if (mode == kMaskVisible)
    launch_bwd_mode<T, DP, kMaskVisible>(p, register_staging, s);
  else if (mode == kMaskBits)
    launch_bwd_mode<T, DP, kMaskBits>(p, register_staging, s);
  else if (mode == kMaskBitsDropout)
    launch_bwd_mode<T, DP, kMaskBitsDropout>(p, register_staging, s);
  else
    launch_bwd_mode<T, DP, kMaskNone>(p, register_staging, s);
}

template <typename T>
void launch_bwd(const AttnBwdParams& p, int mode, bool register_staging, hipStream_t s) {
  if (p.d <= 32)
    launch_bwd_dp<T, 32>(p, mode, register_staging, s);
  else
    launch_bwd_dp<T, 64>(p, mode, register_staging, s);
}

}  // namespace
}  // namespace taac

namespace taac {
namespace {
int attention_bwd_entry(const char* name, const void* q, const void* k, const void* v, const void* o, const void* dout,
                        const float* lse, const int32_t* key_lengths, const uint8_t* drop_mask, float drop_scale, void* dq,
                        void* dk, void* dv, float* delta, int32_t B, int32_t H, int32_t Tq, int32_t Tk, int32_t d,
                        const int64_t q_strides[4], const int64_t k_strides[4], const int64_t v_strides[4],
                        const int64_t o_strides[4], const int64_t do_strides[4], const int64_t dq_strides[4],
                        const int64_t dk_strides[4], const int64_t dv_strides[4], int is_causal, int zero_padded_queries,
                        int dtype, void* stream, int mask_mode = -1, int64_t mask_bs = 0, int64_t mask_hs = 0,
                        const uint8_t* key_valid = nullptr, const uint32_t* bit_words = nullptr, int64_t bits_bs = 0,
                        const int32_t* row_offsets = nullptr) {
  // mask_mode -1: dropout when a mask is given (its matrices follow the (B, H) order), nothing otherwise
  if (mask_mode < 0 || mask_mode == kMaskBitsDropout) {
    if (mask_mode < 0) mask_mode = drop_mask != nullptr ? kMaskDropout : kMaskNone;
    mask_hs = static_cast<int64_t>(Tq) * Tk;
    mask_bs = mask_hs * H;
  }
  if (mask_bs < 0 || mask_hs < 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: negative mask stride", name);
  if (drop_mask != nullptr && !(drop_scale >= 1.f))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: dropout_scale = 1 / (1 - p) must be >= 1", name);
  if (B < 0 || H < 0 || Tq < 0 || Tk < 0 || d <= 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: negative dimension or non-positive head_dim", name);
  if (is_causal & ~(TAAC_ATTN_CAUSAL | TAAC_ATTN_REGISTER_STAGING))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: unknown bits in is_causal (%d)", name, is_causal);
  const bool register_staging = (is_causal & TAAC_ATTN_REGISTER_STAGING) != 0;
  if (dtype != TAAC_BF16 && dtype != TAAC_F16)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: dtype must be bf16 or fp16 (got %d)", name, dtype);
  if (d % 8 != 0 || d > 64)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: head_dim %d unsupported (multiple of 8, at most 64)", name, d);
  if (B == 0 || H == 0 || (Tq == 0 && Tk == 0)) return TAAC_OK;
  if (Tq == 0 || Tk == 0)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: empty query or key sequences are not supported", name);
  if (!q || !k || !v || !o || !dout || !lse || !dq || !dk || !dv || !delta)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: null tensor pointer", name);
  const int64_t* all[8] = {q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides, dk_strides, dv_strides};
  for (const int64_t* st : all)
    if (!strides_ok(st))
      return set_error(TAAC_ERR_UNSUPPORTED,
                       "%s: strides must be non-negative multiples of 8 elements with a unit last stride", name);
  const void* ptrs[8] = {q, k, v, o, dout, dq, dk, dv};
  for (const void* ptr : ptrs)
    if (!aligned16(ptr)) return set_error(TAAC_ERR_UNSUPPORTED, "%s: tensor base pointers must be 16-byte aligned", name);
  if (zero_padded_queries && Tq != Tk)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: zero_padded_queries requires Tq == Tk", name);
  const int64_t blocks = (static_cast<int64_t>(Tq > Tk ? Tq : Tk) + kOwn - 1) / kOwn * B * H;
  if (blocks > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: too many workgroups", name);
  AttnBwdParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  p.dout = dout;
  p.lse = lse;
  p.delta = delta;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.key_lengths = key_lengths;
  p.drop_mask = drop_mask;
  p.mask_bs = mask_bs;
  p.mask_hs = mask_hs;
  p.key_valid = key_valid;
  p.bit_words = bit_words;
  p.bits_bs = bits_bs;
  p.row_offsets = row_offsets;
  p.drop_scale = drop_scale;
  p.B = B;
  p.H = H;
  p.Tq = Tq;
  p.Tk = Tk;
  p.d = d;
  for (int i = 0; i < 4; ++i) {
    p.qs[i] = q_strides[i];
    p.ks[i] = k_strides[i];
    p.vs[i] = v_strides[i];
    p.os[i] = o_strides[i];
    p.dos[i] = do_strides[i];
    p.dqs[i] = dq_strides[i];
    p.dks[i] = dk_strides[i];
    p.dvs[i] = dv_strides[i];
  }
  p.scale = 1.0f / sqrtf(static_cast<float>(d));
  p.zero_pad = zero_padded_queries ? 1 : 0;
  p.causal = (is_causal & TAAC_ATTN_CAUSAL) ? 1 : 0;
  hipStream_t s = as_stream(stream);
  if (dtype == TAAC_BF16)
    launch_bwd<bf16_t>(p, mask_mode, register_staging, s);
  else
    launch_bwd<f16_t>(p, mask_mode, register_staging, s);
  return check_launch(name);
}
}  // namespace
}  // namespace taac

namespace taac {
int attention_compact_bwd(const char* name, const void* qk, const void* v, int64_t ld_qk, int64_t ld_v, const void* o, int64_t ld_o,
                          const void* dout, int64_t ld_do, const float* lse, const int32_t* lengths, const int32_t* row_offsets,
                          const uint32_t* struct_bits, int64_t struct_stride, void* dqkv, int64_t ld_dqkv, float* delta, int32_t B,
                          int32_t H, int32_t T, int32_t dh, hipStream_t s) {
  const int64_t width = static_cast<int64_t>(H) * dh;
  const int64_t qs[4] = {0, dh, ld_qk, 1}, vs[4] = {0, dh, ld_v, 1}, os[4] = {0, dh, ld_o, 1}, dos[4] = {0, dh, ld_do, 1},
                gs[4] = {0, dh, ld_dqkv, 1};
  const bf16_t* q = static_cast<const bf16_t*>(qk);
  bf16_t* g = static_cast<bf16_t*>(dqkv);
  return attention_bwd_entry(name, q, q + width, v, o, dout, lse, lengths, nullptr, 1.f, g, g + width, g + 2 * width, delta, B, H,
                             T, T, dh, qs, qs, vs, os, dos, gs, gs, gs, 0, 1, TAAC_BF16, s,
                             struct_bits != nullptr ? kMaskBits : -1, 0, 0, nullptr, struct_bits, struct_stride, row_offsets);
}
}  // namespace taac

extern "C" int taac_flash_attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                   const float* lse, const int32_t* key_lengths, void* dq, void* dk, void* dv,
                                   float* delta, int32_t B, int32_t H, int32_t Tq, int32_t Tk, int32_t d,
                                   const int64_t q_strides[4], const int64_t k_strides[4], const int64_t v_strides[4],
                                   const int64_t o_strides[4], const int64_t do_strides[4], const int64_t dq_strides[4],
                                   const int64_t dk_strides[4], const int64_t dv_strides[4], int is_causal,
                                   int zero_padded_queries, int dtype, void* stream) {
  return taac::attention_bwd_entry("taac_flash_attn_bwd", q, k, v, o, dout, lse, key_lengths, nullptr, 1.f, dq, dk, dv, delta,
                                   B, H, Tq, Tk, d, q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides,
                                   dk_strides, dv_strides, is_causal, zero_padded_queries, dtype, stream);
}

extern "C" int taac_flash_attn_dropout_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                           const float* lse, const int32_t* key_lengths, const uint8_t* dropout_mask,
                                           float dropout_scale, void* dq, void* dk, void* dv, float* delta, int32_t B,
                                           int32_t H, int32_t Tq, int32_t Tk, int32_t d, const int64_t q_strides[4],
                                           const int64_t k_strides[4], const int64_t v_strides[4],
                                           const int64_t o_strides[4], const int64_t do_strides[4],
                                           const int64_t dq_strides[4], const int64_t dk_strides[4],
                                           const int64_t dv_strides[4], int is_causal, int zero_padded_queries, int dtype,
                                           void* stream) {
  const char* name = "taac_flash_attn_dropout_bwd";
  if (!dropout_mask) return taac::set_error(TAAC_ERR_INVALID_VALUE, "%s: dropout_mask must be given", name);
  return taac::attention_bwd_entry(name, q, k, v, o, dout, lse, key_lengths, dropout_mask, dropout_scale, dq, dk, dv, delta,
                                   B, H, Tq, Tk, d, q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides,
                                   dk_strides, dv_strides, is_causal, zero_padded_queries, dtype, stream);
}

extern "C" int taac_flash_attn_mask_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                        const float* lse, const int32_t* key_lengths, const uint8_t* visible,
                                        int64_t visible_batch_stride, int64_t visible_head_stride,
                                        const uint8_t* key_valid, void* dq, void* dk,
                                        void* dv, float* delta, int32_t B, int32_t H, int32_t Tq, int32_t Tk, int32_t d,
                                        const int64_t q_strides[4], const int64_t k_strides[4], const int64_t v_strides[4],
                                        const int64_t o_strides[4], const int64_t do_strides[4],
                                        const int64_t dq_strides[4], const int64_t dk_strides[4],
                                        const int64_t dv_strides[4], int zero_padded_queries, int dtype, void* stream) {
  const char* name = "taac_flash_attn_mask_bwd";
  if (!visible) return taac::set_error(TAAC_ERR_INVALID_VALUE, "%s: the visibility mask must be given", name);
  return taac::attention_bwd_entry(name, q, k, v, o, dout, lse, key_lengths, visible, 1.f, dq, dk, dv, delta, B, H, Tq, Tk, d,
                                   q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides, dk_strides,
                                   dv_strides, 0, zero_padded_queries, dtype, stream, taac::kMaskVisible,
                                   visible_batch_stride, visible_head_stride, key_valid);
}

extern "C" int taac_flash_attn_bits_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                        const float* lse, const int32_t* key_lengths, const uint32_t* struct_bits,
                                        int64_t struct_sample_stride, const uint32_t* valid_bits,
                                        const uint8_t* dropout_mask, float dropout_scale, void* dq, void* dk, void* dv,
                                        float* delta, int32_t B, int32_t H, int32_t Tq, int32_t Tk, int32_t d,
                                        const int64_t q_strides[4], const int64_t k_strides[4], const int64_t v_strides[4],
                                        const int64_t o_strides[4], const int64_t do_strides[4],
                                        const int64_t dq_strides[4], const int64_t dk_strides[4],
                                        const int64_t dv_strides[4], int zero_padded_queries, int dtype, void* stream) {
  const char* name = "taac_flash_attn_bits_bwd";
  if (!struct_bits) return taac::set_error(TAAC_ERR_INVALID_VALUE, "%s: struct_bits must be given", name);
  if (struct_sample_stride < 0) return taac::set_error(TAAC_ERR_INVALID_VALUE, "%s: negative sample stride", name);
  return taac::attention_bwd_entry(name, q, k, v, o, dout, lse, key_lengths, dropout_mask,
                                   dropout_mask != nullptr ? dropout_scale : 1.f, dq, dk, dv, delta, B, H, Tq, Tk, d,
                                   q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides, dk_strides,
                                   dv_strides, 0, zero_padded_queries, dtype, stream,
                                   dropout_mask != nullptr ? taac::kMaskBitsDropout : taac::kMaskBits, 0, 0,
                                   reinterpret_cast<const uint8_t*>(valid_bits), struct_bits, struct_sample_stride);
}
