// Forward driver of the unified token backbone (pre-norm blocks + pCVR readout) and the readout kernel.
// The driver only sequences the library's own entry points on one stream over a caller-provided workspace.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "common.h"
#include "row_index.h"

namespace taac {
namespace {

constexpr int kBlock = 256;

inline int64_t align256(int64_t v) { return (v + 255) & ~static_cast<int64_t>(255); }

// One workgroup per sample: fp32 sum over the valid prefix of the sample's tokens, mean, dot with the head weight,
// sigmoid. Thread layout: chunk = tid % (D/8) picks 8 features, group = tid / (D/8) strides over tokens.
__global__ __launch_bounds__(kBlock) void masked_mean_head_kernel(const bf16_t* __restrict__ x,
                                                                  const int32_t* __restrict__ lengths,
                                                                  const bf16_t* __restrict__ w_head,
                                                                  const bf16_t* __restrict__ b_head,
                                                                  float* __restrict__ p, int T, int D) {
  __shared__ float s_acc[kBlock][8];
  __shared__ float s_dot[kBlock];
  const int b = blockIdx.x;
  const int c8n = D / 8;
  const int groups = kBlock / c8n;
  const int chunk = threadIdx.x % c8n;
  const int group = threadIdx.x / c8n;
  int len = lengths[b];
  len = len < 0 ? 0 : (len > T ? T : len);
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  if (group < groups) {
    const bf16_t* xb = x + static_cast<int64_t>(b) * T * D + chunk * 8;
    for (int t = group; t < len; t += groups) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(xb + static_cast<int64_t>(t) * D);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += static_cast<float>(v[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s_acc[threadIdx.x][e] = acc[e];
  __syncthreads();
  float dot = 0.f;
  if (threadIdx.x < c8n) {
    const float denom = static_cast<float>(len < 1 ? 1 : len);
    const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w_head + threadIdx.x * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float s = 0.f;
      for (int g = 0; g < groups; ++g) s += s_acc[g * c8n + threadIdx.x][e];
      dot += (s / denom) * static_cast<float>(wv[e]);
    }
  }
  s_dot[threadIdx.x] = dot;
  __syncthreads();
  if (threadIdx.x == 0) {
    float z = b_head != nullptr ? static_cast<float>(b_head[0]) : 0.f;
    for (int i = 0; i < c8n; ++i) z += s_dot[i];
    p[b] = 1.0f / (1.0f + expf(-z));
  }
}

// The same readout from per-token dot products with the head weight (left behind by the last block's kernel): one
// wavefront per sample adds the dots of its valid prefix in a fixed order, mean, bias, sigmoid.
__global__ __launch_bounds__(kBlock) void token_dots_head_kernel(const float* __restrict__ dots,
                                                                 const int32_t* __restrict__ lengths,
                                                                 const bf16_t* __restrict__ b_head, float* __restrict__ p,
                                                                 int B, int T) {
  const int b = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  if (b >= B) return;
  int len = lengths[b];
  len = len < 0 ? 0 : (len > T ? T : len);
  const float* row = dots + static_cast<int64_t>(b) * T;
  float s = 0.f;
  for (int t = lane; t < len; t += kWave) s += row[t];
  s = group_sum<kWave>(s);
  if (lane == 0) {
    const float z = (b_head != nullptr ? static_cast<float>(b_head[0]) : 0.f) + s / static_cast<float>(len < 1 ? 1 : len);
    p[b] = 1.0f / (1.0f + expf(-z));
  }
}

// Batches too large for one launch (row_index.h): exclusive prefix sums of the per-sample valid counts (one workgroup; B is walked
// in slabs of kBlock with a running carry), then the rows (valid_rows_kernel / valid_rows_bits_kernel).
__global__ __launch_bounds__(kBlock) void length_offsets_kernel(const int32_t* __restrict__ lengths,
                                                                const uint32_t* __restrict__ bits, int B, int T,
                                                                int32_t* __restrict__ offsets,
                                                                int32_t* __restrict__ n_rows) {
  __shared__ int32_t s_scan[kBlock];
  int32_t carry = 0;
  for (int base = 0; base < B; base += kBlock) {
    const int b = base + threadIdx.x;
    const int32_t len = b >= B ? 0 : (lengths != nullptr ? clamped_length(lengths, b, T) : valid_bit_count(bits, b, T));
    s_scan[threadIdx.x] = len;
    __syncthreads();
    for (int step = 1; step < kBlock; step <<= 1) {  // inclusive scan, Hillis-Steele
      const int32_t add = threadIdx.x >= step ? s_scan[threadIdx.x - step] : 0;
      __syncthreads();
      s_scan[threadIdx.x] += add;
      __syncthreads();
    }
    if (b < B) offsets[b] = carry + s_scan[threadIdx.x] - len;
    carry += s_scan[kBlock - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    offsets[B] = carry;
    *n_rows = carry;
  }
}

__global__ __launch_bounds__(kBlock) void valid_rows_kernel(const int32_t* __restrict__ lengths,
                                                            const int32_t* __restrict__ offsets, int T,
                                                            int32_t* __restrict__ rows) {
  const int b = blockIdx.y;
  int32_t len = lengths[b];
  len = len < 0 ? 0 : (len > T ? T : len);
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t < len) rows[offsets[b] + t] = b * T + t;
}

// The same for a validity bit row per sample: token t goes to slot offsets[b] + (number of valid tokens before t).
__global__ __launch_bounds__(kBlock) void valid_rows_bits_kernel(const uint32_t* __restrict__ bits,
                                                                 const int32_t* __restrict__ offsets, int T,
                                                                 int32_t* __restrict__ rows) {
  const int b = blockIdx.y;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= T) return;
  const int wpr = (T + 31) / 32;
  const uint32_t* row = bits + static_cast<int64_t>(b) * wpr;
  const uint32_t word = row[t / 32];
  if (((word >> (t % 32)) & 1u) == 0u) return;
  int32_t rank = __popc(word & ((1u << (t % 32)) - 1u));
  for (int w = 0; w < t / 32; ++w) rank += __popc(row[w]);
  rows[offsets[b] + rank] = b * T + t;
}

// The index in one launch (see row_index.h).
__global__ __launch_bounds__(kRowThreads) void valid_rows_scan_kernel(const int32_t* __restrict__ lengths, int B, int T,
                                                                      int32_t* __restrict__ rows, int32_t* __restrict__ n_rows) {
  write_valid_rows(lengths, B, T, blockIdx.x, rows, n_rows);
}
__global__ __launch_bounds__(kRowThreads) void valid_rows_bits_scan_kernel(const uint32_t* __restrict__ bits, int B, int T,
                                                                           int32_t* __restrict__ rows,
                                                                           int32_t* __restrict__ n_rows) {
  write_valid_rows_bits(bits, B, T, blockIdx.x, rows, n_rows);
}

// front_rows[i] = b * T + (i - offsets[b]) for token i of sample b = rows[i] / T; lengths[b] = offsets[b + 1] - offsets[b].
__global__ __launch_bounds__(kBlock) void front_rows_kernel(const int32_t* __restrict__ rows,
                                                            const int32_t* __restrict__ n_rows, int B, int T,
                                                            int32_t* __restrict__ front_rows,
                                                            int32_t* __restrict__ lengths) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  const int32_t* offsets = rows + static_cast<int64_t>(B) * T;
  if (i < B) lengths[i] = offsets[i + 1] - offsets[i];
  if (i >= *n_rows) return;
  const int b = rows[i] / T;
  front_rows[i] = b * T + static_cast<int32_t>(i - offsets[b]);
}

// One workgroup per (sample b, kFrontRowsPerBlock front rows). The front keys are the sample's valid positions in ascending order, so a
// front row is its structure row with the bits of the invalid positions squeezed out: one lane takes a word of 32 positions, moves each
// kept bit down by the number of dropped ones below it - by 1, 2, 4, 8 and 16 where that number has the digit ("compress" in
// H. S. Warren, Hacker's Delight, 2nd edition, section 7-4); which bits move in which
// step depends on the validity word alone, so a lane works it out once for all its rows - and ORs the piece into the row's words
// in LDS from the bit on at which the valid positions in front of the word end. An index that lists a sample's positions in another
// order is gathered bit by bit (nothing in this library makes one; the look at the order is up to 0.4 us, 512 x 403). Only rows below the sample's number of valid tokens n_b are written,
// and of those the words that hold a key below n_b's 64-key group (the attention kernel reads nothing else), bits at or beyond n_b as zeros.
// Bound by the chain of loads in front of it (offsets, positions, structure words). Before, a lane picked the word of its key by a
// lane permute and a ballot gathered 64 bits. Before / now, us, samples x positions, 30 % of them invalid: 16 x 403 6.2 / 3.7,
// 512 x 403 23.1 / 11.3 (none invalid 36.3 / 16.1, 80 % 7.8 / 6.8), 512 x 200 10.5 / 7.5, 64 x 2048 60.9 / 20.6, 32 x 4096
// 105.5 / 39.3. Rows of a workgroup: 32 / 64 / 128, 512 x 403 16.0 / 11.3 / 12.6, 16 x 403 3.6 / 3.7 / 4.6, 32 x 4096 37.4 / 39.3 / 44.9.
constexpr int kFrontRowsPerBlock = 64;
constexpr int kFrontWords = 4096 / 32;
constexpr int kFrontRowsAtOnce = 4;
__global__ __launch_bounds__(kBlock) void mask_front_bits_kernel(const uint32_t* __restrict__ struct_bits, int T,
                                                                 const int32_t* __restrict__ rows, int B,
                                                                 uint32_t* __restrict__ out) {
  __shared__ uint32_t valid[kFrontWords];
  __shared__ uint32_t position[kFrontRowsPerBlock], descends;
  extern __shared__ uint32_t front[];  // [kFrontRowsPerBlock][wpr]
  const int wpr = (T + 31) / 32;
  const int slabs = (T + kFrontRowsPerBlock - 1) / kFrontRowsPerBlock;
  const int b = blockIdx.x / slabs, r0 = (blockIdx.x % slabs) * kFrontRowsPerBlock;
  const int32_t* offsets = rows + static_cast<int64_t>(B) * T;
  const int32_t off = offsets[b];
  const int n = offsets[b + 1] - off;
  if (r0 >= n) return;  // workgroup-uniform
  const int here = n - r0 < kFrontRowsPerBlock ? n - r0 : kFrontRowsPerBlock;
  if (threadIdx.x < kFrontWords) valid[threadIdx.x] = 0u;
  if (threadIdx.x == 0) descends = 0u;
  for (int i = threadIdx.x; i < here * wpr; i += kBlock) front[i] = 0u;
  __syncthreads();
  const int written = (n + kWave - 1) / kWave * 2 < wpr ? (n + kWave - 1) / kWave * 2 : wpr;
  for (int j = threadIdx.x; j < n; j += kBlock) {
    const int32_t row = rows[off + j];
    if (j + 1 < n && row >= rows[off + j + 1]) descends = 1u;
    const uint32_t at = static_cast<uint32_t>(row - b * T);
    if (at < static_cast<uint32_t>(T)) atomicOr(&valid[at / 32], 1u << (at % 32));
    if (j >= r0 && j < r0 + here) position[j - r0] = at < static_cast<uint32_t>(T) ? at : 0u;
  }
  __syncthreads();
  if (descends != 0u) {
    for (int i = threadIdx.x; i < here * written; i += kBlock) {
      const int r = i / written, first = i % written * 32;
      uint32_t bits = 0u;
      for (int k = 0; k < 32 && first + k < n; ++k) {
        const uint32_t at = static_cast<uint32_t>(rows[off + first + k] - b * T);
        if (at < static_cast<uint32_t>(T)) bits |= ((struct_bits[static_cast<int64_t>(position[r]) * wpr + at / 32] >> (at % 32)) & 1u) << k;
      }
      out[(static_cast<int64_t>(b) * T + r0 + r) * wpr + first / 32] = bits;
    }
    return;
  }
  // lanes of a row: wpr rounded up to a power of two
  const int shift = wpr <= 1 ? 0 : 32 - __builtin_clz(static_cast<unsigned>(wpr - 1));
  const int word = threadIdx.x & ((1 << shift) - 1), row0 = threadIdx.x >> shift, rows_at_once = kBlock >> shift;
  uint32_t words[kFrontRowsAtOnce];
  auto request = [&](int first) {
#pragma unroll
    for (int i = 0; i < kFrontRowsAtOnce; ++i) {
      const int r = first + i * rows_at_once;
      words[i] = (word < wpr && r < here) ? struct_bits[static_cast<int64_t>(position[r]) * wpr + word] : 0u;
    }
  };
  request(row0);
  // valid positions in front of the lane's word: every wavefront scans all words, two a lane
  const int lane = threadIdx.x % kWave;
  const int even = __popc(valid[2 * lane]);
  int upto = even + __popc(valid[2 * lane + 1]);
  const int pair = upto;
#pragma unroll
  for (int step = 1; step < kWave; step <<= 1) {
    const int below = __shfl_up(upto, step, kWave);
    if (lane >= step) upto += below;
  }
  const int pairs_before = __shfl(upto - pair, word / 2, kWave), even_before = __shfl(even, word / 2, kWave);
  const int before = pairs_before + ((word & 1) ? even_before : 0);
  // moved[k]: the bits that move down by 2^k. `odd`: at each bit, whether the number of dropped bits below it that are still to
  // be counted is odd; those at odd counts are then taken out, which halves the counts for the next step.
  const uint32_t keep = valid[word];
  uint32_t moved[5], kept = keep, dropped_below = ~keep << 1;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    uint32_t odd = dropped_below;
#pragma unroll
    for (int step = 1; step < 32; step <<= 1) odd ^= odd << step;
    moved[k] = odd & kept;
    kept = (kept ^ moved[k]) | (moved[k] >> (1 << k));
    dropped_below &= ~odd;
  }
  for (int first = row0; first < here; first += kFrontRowsAtOnce * rows_at_once) {
    if (first != row0) request(first);
#pragma unroll
    for (int i = 0; i < kFrontRowsAtOnce; ++i) {
      const int r = first + i * rows_at_once;
      uint32_t bits = words[i] & keep;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const uint32_t moving = bits & moved[k];
        bits = (bits ^ moving) | (moving >> (1 << k));
      }
      const uint64_t piece = static_cast<uint64_t>(bits) << (before % 32);
      const uint32_t lo = static_cast<uint32_t>(piece), hi = static_cast<uint32_t>(piece >> 32);
      uint32_t* dst = front + r * wpr + before / 32;
      if (lo != 0u) atomicOr(dst, lo);  // a bit that is set stands for a key below n: within the row's words
      if (hi != 0u) atomicOr(dst + 1, hi);
    }
  }
  __syncthreads();
  if (word < written)
    for (int r = row0; r < here; r += rows_at_once)
      out[(static_cast<int64_t>(b) * T + r0 + r) * wpr + word] = front[r * wpr + word];
}

}  // namespace
}  // namespace taac

namespace taac {
namespace {
// One 16-byte piece per thread: row (b, t) of out is a[offsets[b] + t] (+ b2 of the same row) when t < lengths[b], else
// the row of `padded`.
__global__ __launch_bounds__(kBlock) void rows_merge_kernel(const bf16x8* __restrict__ padded, const bf16x8* __restrict__ a,
                                                            const bf16x8* __restrict__ b2,
                                                            const int32_t* __restrict__ lengths,
                                                            const int32_t* __restrict__ offsets, bf16x8* __restrict__ out,
                                                            int64_t pieces_total, int T, int pieces) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (idx >= pieces_total) return;
  const int64_t row = idx / pieces;
  const int c = static_cast<int>(idx % pieces);
  const int b = static_cast<int>(row / T), t = static_cast<int>(row % T);
  int32_t len = lengths[b];
  len = len < 0 ? 0 : (len > T ? T : len);
  bf16x8 v;
  if (t < len) {
    const int64_t src = (static_cast<int64_t>(offsets[b]) + t) * pieces + c;
    v = a[src];
    if (b2 != nullptr) {
      const bf16x8 w = b2[src];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) + static_cast<float>(w[e]));
    }
  } else {
    v = padded[idx];
  }
  out[idx] = v;
}

// The same merge for padding that is not a prefix: (b, t) is valid iff bit t of valid_bits[b] is set, and its compact row
// is offsets[b] + the number of valid tokens of the sample in front of it (word_prefix[b][w], if given, = the number of
// valid tokens in the words before word w, which saves the walk over those words).
__global__ __launch_bounds__(kBlock) void rows_merge_bits_kernel(const bf16x8* __restrict__ padded,
                                                                 const bf16x8* __restrict__ a, const bf16x8* __restrict__ b2,
                                                                 const uint32_t* __restrict__ valid_bits,
                                                                 const int32_t* __restrict__ word_prefix,
                                                                 const int32_t* __restrict__ offsets, bf16x8* __restrict__ out,
                                                                 int64_t pieces_total, int T, int pieces) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (idx >= pieces_total) return;
  const int64_t row = idx / pieces;
  const int c = static_cast<int>(idx % pieces);
  const int b = static_cast<int>(row / T), t = static_cast<int>(row % T);
  const uint32_t* bits = valid_bits + static_cast<int64_t>(b) * ((T + 31) / 32);
  const uint32_t word = bits[t / 32];
  bf16x8 v;
  if ((word >> (t % 32)) & 1u) {
    int rank = __popc(word & ((1u << (t % 32)) - 1u));
    if (word_prefix != nullptr) {
      rank += word_prefix[static_cast<int64_t>(b) * ((T + 31) / 32) + t / 32];
    } else {
      for (int w = 0; w < t / 32; ++w) rank += __popc(bits[w]);
    }
    const int64_t src = (static_cast<int64_t>(offsets[b]) + rank) * pieces + c;
    v = a[src];
    if (b2 != nullptr) {
      const bf16x8 w2 = b2[src];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16_t>(static_cast<float>(v[e]) + static_cast<float>(w2[e]));
    }
  } else {
    v = padded[idx];
  }
  out[idx] = v;
}

// dst[i] = src[rows[i]] for i < n: one 16-byte piece per thread.
__global__ __launch_bounds__(kBlock) void rows_gather_kernel(const bf16x8* __restrict__ src, int64_t src_pieces,
                                                             const int32_t* __restrict__ rows, bf16x8* __restrict__ dst,
                                                             int64_t pieces_total, int pieces) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (idx >= pieces_total) return;
  const int64_t i = idx / pieces;
  const int c = static_cast<int>(idx % pieces);
  dst[idx] = __builtin_nontemporal_load(src + static_cast<int64_t>(rows[i]) * src_pieces + c);
}
}  // namespace
}  // namespace taac

extern "C" int taac_rows_gather(const void* src, int64_t ld_src, const int32_t* rows, int64_t n, void* dst, int32_t W,
                                void* stream) {
  using namespace taac;
  const char* name = "taac_rows_gather";
  if (n < 0 || W <= 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (W % 8 != 0 || ld_src % 8 != 0 || ld_src < W)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: W and the source row stride must be multiples of 8 and cover a row", name);
  if (n == 0) return TAAC_OK;
  if (!src || !rows || !dst) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(src) || !aligned16(dst)) return set_error(TAAC_ERR_UNSUPPORTED, "%s: tensor base pointers must be 16-byte aligned", name);
  const int64_t pieces_total = n * (W / 8);
  const int64_t blocks = (pieces_total + kBlock - 1) / kBlock;
  if (blocks > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: too many workgroups", name);
  hipLaunchKernelGGL(rows_gather_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kBlock), 0, as_stream(stream),
                     static_cast<const bf16x8*>(src), ld_src / 8, rows, static_cast<bf16x8*>(dst), pieces_total, W / 8);
  return check_launch(name);
}

extern "C" int taac_rows_merge(const void* padded, const void* compact_a, const void* compact_b, const int32_t* key_lengths,
                               const int32_t* offsets, void* out, int32_t B, int32_t T, int32_t W, void* stream) {
  using namespace taac;
  const char* name = "taac_rows_merge";
  if (B < 0 || T < 0 || W <= 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (W % 8 != 0) return set_error(TAAC_ERR_UNSUPPORTED, "%s: W=%d must be a multiple of 8", name, W);
  if (B == 0 || T == 0) return TAAC_OK;
  if (!padded || !compact_a || !key_lengths || !offsets || !out) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(padded) || !aligned16(compact_a) || !aligned16(compact_b) || !aligned16(out))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: tensor base pointers must be 16-byte aligned", name);
  const int64_t pieces_total = static_cast<int64_t>(B) * T * (W / 8);
  const int64_t blocks = (pieces_total + kBlock - 1) / kBlock;
  if (blocks > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: too many workgroups", name);
  hipLaunchKernelGGL(rows_merge_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kBlock), 0, as_stream(stream),
                     static_cast<const bf16x8*>(padded), static_cast<const bf16x8*>(compact_a),
                     static_cast<const bf16x8*>(compact_b), key_lengths, offsets, static_cast<bf16x8*>(out), pieces_total, T,
                     W / 8);
  return check_launch(name);
}

extern "C" int taac_rows_merge_bits(const void* padded, const void* compact_a, const void* compact_b,
                                    const uint32_t* valid_bits, const int32_t* word_prefix, const int32_t* offsets,
                                    void* out, int32_t B, int32_t T, int32_t W, void* stream) {
  using namespace taac;
  const char* name = "taac_rows_merge_bits";
  if (B < 0 || T < 0 || W <= 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (W % 8 != 0) return set_error(TAAC_ERR_UNSUPPORTED, "%s: W=%d must be a multiple of 8", name, W);
  if (B == 0 || T == 0) return TAAC_OK;
  if (!padded || !compact_a || !valid_bits || !offsets || !out) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(padded) || !aligned16(compact_a) || !aligned16(compact_b) || !aligned16(out))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: tensor base pointers must be 16-byte aligned", name);
  const int64_t pieces_total = static_cast<int64_t>(B) * T * (W / 8);
  const int64_t blocks = (pieces_total + kBlock - 1) / kBlock;
  if (blocks > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: too many workgroups", name);
  hipLaunchKernelGGL(rows_merge_bits_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kBlock), 0, as_stream(stream),
                     static_cast<const bf16x8*>(padded), static_cast<const bf16x8*>(compact_a),
                     static_cast<const bf16x8*>(compact_b), valid_bits, word_prefix, offsets, static_cast<bf16x8*>(out),
                     pieces_total, T, W / 8);
  return check_launch(name);
}

extern "C" int taac_valid_rows(const int32_t* key_lengths, int32_t B, int32_t T, int32_t* rows, int32_t* n_rows,
                               void* stream) {
  using namespace taac;
  const char* name = "taac_valid_rows";
  if (B < 0 || T < 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (static_cast<int64_t>(B) * T > 0x7fffffffLL - B - 1)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: B * T must fit 32-bit row numbers", name);
  if (!rows || !n_rows || (B > 0 && !key_lengths)) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (B > 65535) return set_error(TAAC_ERR_UNSUPPORTED, "%s: at most 65535 samples", name);
  if (B > 0 && T > 0 && row_index_in_one_launch(B, T, false)) {
    const uint32_t units = static_cast<uint32_t>(B) * ((T + kRowThreads - 1) / kRowThreads);
    hipLaunchKernelGGL(valid_rows_scan_kernel, dim3(units), dim3(kRowThreads), 0, as_stream(stream), key_lengths, B, T, rows, n_rows);
    return check_launch(name);
  }
  int32_t* offsets = rows + static_cast<int64_t>(B) * T;
  hipLaunchKernelGGL(length_offsets_kernel, dim3(1), dim3(kBlock), 0, as_stream(stream), key_lengths,
                     static_cast<const uint32_t*>(nullptr), B, T, offsets, n_rows);
  if (B > 0 && T > 0)
    hipLaunchKernelGGL(valid_rows_kernel, dim3((T + kBlock - 1) / kBlock, B), dim3(kBlock), 0, as_stream(stream),
                       key_lengths, offsets, T, rows);
  return check_launch(name);
}

extern "C" int taac_valid_rows_from_bits(const uint32_t* valid_bits, int32_t B, int32_t T, int32_t* rows,
                                         int32_t* n_rows, void* stream) {
  using namespace taac;
  const char* name = "taac_valid_rows_from_bits";
  if (B < 0 || T < 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (static_cast<int64_t>(B) * T > 0x7fffffffLL - B - 1)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: B * T must fit 32-bit row numbers", name);
  if (!rows || !n_rows || (B > 0 && T > 0 && !valid_bits)) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (B > 65535) return set_error(TAAC_ERR_UNSUPPORTED, "%s: at most 65535 samples", name);
  if (B > 0 && T > 0 && row_index_in_one_launch(B, T, true)) {
    const uint32_t units = static_cast<uint32_t>(B) * ((T + kRowThreads - 1) / kRowThreads);
    hipLaunchKernelGGL(valid_rows_bits_scan_kernel, dim3(units), dim3(kRowThreads), 0, as_stream(stream), valid_bits, B, T, rows, n_rows);
    return check_launch(name);
  }
  int32_t* offsets = rows + static_cast<int64_t>(B) * T;
  hipLaunchKernelGGL(length_offsets_kernel, dim3(1), dim3(kBlock), 0, as_stream(stream),
                     static_cast<const int32_t*>(nullptr), valid_bits, B, T, offsets, n_rows);
  if (B > 0 && T > 0)
    hipLaunchKernelGGL(valid_rows_bits_kernel, dim3((T + kBlock - 1) / kBlock, B), dim3(kBlock), 0, as_stream(stream),
                       valid_bits, offsets, T, rows);
  return check_launch(name);
}

extern "C" int taac_masked_mean_head(const void* x, const int32_t* lengths, const void* w_head, const void* b_head,
                                     float* p, int32_t B, int32_t T, int32_t D, void* stream) {
  using namespace taac;
  const char* name = "taac_masked_mean_head";
  if (B < 0 || T < 0 || D <= 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (D % 8 != 0 || D > 8 * kBlock)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: D=%d must be a multiple of 8 and at most %d", name, D, 8 * kBlock);
  if (B == 0) return TAAC_OK;
  if (!x || !lengths || !w_head || !p) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(x) || !aligned16(w_head))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: x and w_head must be 16-byte aligned", name);
  hipLaunchKernelGGL(masked_mean_head_kernel, dim3(B), dim3(kBlock), 0, as_stream(stream),
                     static_cast<const bf16_t*>(x), lengths, static_cast<const bf16_t*>(w_head),
                     static_cast<const bf16_t*>(b_head), p, T, D);
  return check_launch(name);
}

namespace taac {
namespace {
// Fused (token-stationary) path: model widths 128 / 256, hidden size a multiple of 32.
inline bool fused_shape(int32_t D, int32_t F) { return (D == 128 || D == 256) && F % 32 == 0; }
// Fragment-ordered weights of one block: qkv, out, feed-forward.
// Row index of the valid tokens: B*T rows + B+1 offsets + the count.
inline int64_t row_index_bytes(int32_t B, int32_t T) { return align256((static_cast<int64_t>(B) * T + B + 2) * 4); }
inline int64_t packed_block_bytes(int32_t D, int32_t F) {
  return align256(static_cast<int64_t>(3) * D * D * 2) + align256(static_cast<int64_t>(D) * D * 2) +
         align256(static_cast<int64_t>(3) * D * F * 2);
}
// Query / key norm scratch of the fused path: per-chunk sums of squares [2D / 64, M] and the counters behind them, factors [2, M], per
// block the product of the query and key norm weights (fp32 [D]) or, with a rotary table, the two weights side by side (bf16 [2D]).
inline int64_t qk_sums_bytes(int64_t M, int32_t D) { return align256((2 * D / 64) * M * 4); }
inline int64_t qk_norm_bytes(int64_t M, int32_t D, int32_t n_blocks) {
  return qk_sums_bytes(M, D) + align256(kQkCounters * 4) + align256(2 * M * 4) + align256(static_cast<int64_t>(D) * 4 * n_blocks);
}
// FP8 mode (TAAC_BACKBONE_FP8; D = 256, F a multiple of 64): per block the e4m3 qkv / out weights, the packed feed-forward
// blob and 8 scales (weights: qkv, out, up, down; activations: block input, attention output, feed-forward input, gated
// hidden state); one more set of scales behind the last block.
inline bool fp8_shape(int32_t D, int32_t F) { return D == 256 && F % 64 == 0; }
inline int64_t fp8_block_bytes(int32_t D, int32_t F) {
  return align256(static_cast<int64_t>(3) * D * D) + align256(static_cast<int64_t>(D) * D) +
         align256(taac_ffn_fp8_packed_bytes(D, F));
}
inline int64_t fp8_bytes(int32_t D, int32_t F, int32_t n_blocks) {
  return fp8_shape(D, F) ? n_blocks * fp8_block_bytes(D, F) + align256((n_blocks + 1) * 8 * 4) : 0;
}
}  // namespace
}  // namespace taac

extern "C" int64_t taac_backbone_workspace_bytes(int32_t B, int32_t T, int32_t D, int32_t F, int32_t n_blocks) {
  using namespace taac;
  if (B < 0 || T < 0 || D <= 0 || F <= 0 || n_blocks < 0) return -1;
  const int64_t M = static_cast<int64_t>(B) * T;
  // x, h (shared with the attention output), qkv, then either the packed weights + the valid-row index (fused path)
  // or the gated hidden state
  const int64_t acts = align256(M * D * 2) * 2 + align256(M * 3 * D * 2);
  return acts + (fused_shape(D, F) ? n_blocks * packed_block_bytes(D, F) + row_index_bytes(B, T) + qk_norm_bytes(M, D, n_blocks) +
                                         align256(ffn_split_bytes(M, D, F)) + fp8_bytes(D, F, n_blocks)
                                   : align256(M * F * 2));
}

extern "C" int64_t taac_backbone_fp8_scales_offset(int32_t B, int32_t T, int32_t D, int32_t F, int32_t n_blocks) {
  using namespace taac;
  if (B < 0 || T < 0 || n_blocks < 0 || !fp8_shape(D, F)) return -1;
  return taac_backbone_workspace_bytes(B, T, D, F, n_blocks) - align256((n_blocks + 1) * 8 * 4);
}

extern "C" int taac_backbone_fwd(const void* emb, const int32_t* key_lengths, const taac_block_weights* blocks,
                                 int32_t n_blocks, const void* w_head, const void* b_head, int32_t B, int32_t T,
                                 int32_t D, int32_t heads, int32_t F, float eps, const void* rope_cos_sin,
                                 int flags, void* workspace, int64_t workspace_bytes, void* hidden_out, float* p,
                                 void* stream) {
  using namespace taac;
  const char* name = "taac_backbone_fwd";
  if (flags & ~(TAAC_BACKBONE_DENSE_TOKENS | TAAC_BACKBONE_SPLIT_OUT_FFN | TAAC_BACKBONE_FP8 | TAAC_BACKBONE_ROW_MAJOR_QKV))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: unknown flag bits (%d)", name, flags);
  const bool fp8 = (flags & TAAC_BACKBONE_FP8) != 0;
  if (fp8 && !fp8_shape(D, F))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: the FP8 dense layers are built for D = 256 and F a multiple of 64", name);
  if (fp8 && rope_cos_sin != nullptr)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: the FP8 mode covers the plain attention layer (no rotary embedding)", name);
  if (B < 0 || T < 0 || D <= 0 || F <= 0 || heads <= 0 || n_blocks < 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (D % heads != 0 || (D / heads) % 8 != 0 || D / heads > 128)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: D=%d heads=%d: head_dim must be a multiple of 8, at most 128", name, D,
                     heads);
  if (D % 8 != 0 || F % 8 != 0) return set_error(TAAC_ERR_UNSUPPORTED, "%s: D and F must be multiples of 8", name);
  if (B == 0 || T == 0) return TAAC_OK;
  if (!emb || !key_lengths || !p || !w_head || (n_blocks > 0 && !blocks))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  const int64_t need = taac_backbone_workspace_bytes(B, T, D, F, n_blocks);
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 255u))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: workspace must be 256-byte aligned and hold %lld bytes", name,
                     (long long)need);

  const int64_t M = static_cast<int64_t>(B) * T;
  char* ws = static_cast<char*>(workspace);
  bf16_t* x = reinterpret_cast<bf16_t*>(ws);
  ws += align256(M * D * 2);
  bf16_t* h = reinterpret_cast<bf16_t*>(ws);
  ws += align256(M * D * 2);
  bf16_t* qkv = reinterpret_cast<bf16_t*>(ws);
  ws += align256(M * 3 * D * 2);
  bf16_t* g = reinterpret_cast<bf16_t*>(ws);  // unfused path: gated hidden state; fused path: packed weights
  char* packed = ws;
  const bool fused = fused_shape(D, F);
  // the packed up projection carries the constants of the gate's activation where the kernels take them from there
  const bool fold_act = fused && ffn_act_fold_supported(D, F);
  // Fused path: the dense layers walk the valid tokens only (row index built from key_lengths on the device); the
  // padded positions of the residual stream are never read or written. TAAC_BACKBONE_DENSE_TOKENS switches this off.
  int32_t* rows = nullptr;
  int32_t* n_rows = nullptr;
  char* after_packed = packed + static_cast<int64_t>(n_blocks) * packed_block_bytes(D, F);
  float* qk_sumsq = reinterpret_cast<float*>(after_packed + row_index_bytes(B, T));
  uint32_t* qk_counters = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(qk_sumsq) + qk_sums_bytes(M, D));
  float* qk_rstd = reinterpret_cast<float*>(reinterpret_cast<char*>(qk_counters) + align256(kQkCounters * 4));
  bf16_t* qk_weight = reinterpret_cast<bf16_t*>(reinterpret_cast<char*>(qk_rstd) + align256(2 * M * 4));
  if (rope_cos_sin != nullptr && !aligned16(rope_cos_sin))
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: the rotary table must be 16-byte aligned", name);
  const bool sparse = fused && n_blocks > 0 && !(flags & TAAC_BACKBONE_DENSE_TOKENS);
  if (sparse) {
    if (M > 0x7fffffffLL - B - 1 || B > 65535)
      return set_error(TAAC_ERR_UNSUPPORTED, "%s: the row index covers at most 65535 samples and 2^31 rows", name);
    rows = reinterpret_cast<int32_t*>(after_packed);
    n_rows = rows + M + B + 1;
  }

  const int dh = D / heads;
  const int64_t qkv_strides[4] = {static_cast<int64_t>(T) * 3 * D, dh, 3 * static_cast<int64_t>(D), 1};
  const int64_t o_strides[4] = {static_cast<int64_t>(T) * D, dh, D, 1};

  const bf16_t* cur = static_cast<const bf16_t*>(emb);
  int rc;
  // TAAC_BACKBONE_SPLIT_OUT_FFN: the out projection and the feed-forward half as two kernels (comparison route).
  const bool split_out_ffn = (flags & TAAC_BACKBONE_SPLIT_OUT_FFN) != 0;
  float* norm_product = reinterpret_cast<float*>(qk_weight);  // [n_blocks, D]
  // partials and counters of a feed-forward whose token tiles are shared by several workgroups (small batches)
  const int ffn_split = fused ? ffn_splits(M, D, F) : 1;
  char* split_scratch = ffn_split > 1 ? reinterpret_cast<char*>(norm_product) + align256(static_cast<int64_t>(D) * 4 * n_blocks) : nullptr;
  const int64_t tiles = (M + 31) / 32;
  uint32_t* split_counters =
      split_scratch != nullptr ? reinterpret_cast<uint32_t*>(split_scratch + tiles * ffn_split * 32 * D * 4) : nullptr;
  if (fused && n_blocks > 0) {
    // One launch: the weights of all blocks in fragment order (the FP8 mode packs its own), the row index, the products of the
    // query and key norm weights, zeros in the padded rows of the returned hidden state.
    std::vector<void*> pk(3 * static_cast<size_t>(n_blocks));
    bool qk_norms = false;
    for (int i = 0; i < n_blocks; ++i) {
      const taac_block_weights& w = blocks[i];
      if (!w.qkv_weight || !w.out_weight || !w.up_weight || !w.down_weight)
        return set_error(TAAC_ERR_INVALID_VALUE, "%s: block %d has a null weight", name, i);
      if ((w.query_norm_weight == nullptr) != (w.key_norm_weight == nullptr))
        return set_error(TAAC_ERR_INVALID_VALUE, "%s: block %d: query and key norm weights come together", name, i);
      qk_norms = qk_norms || w.query_norm_weight != nullptr;
      char* base = packed + static_cast<int64_t>(i) * packed_block_bytes(D, F);
      pk[i] = base;
      pk[n_blocks + i] = base + align256(static_cast<int64_t>(3) * D * D * 2);
      pk[2 * n_blocks + i] = base + align256(static_cast<int64_t>(3) * D * D * 2) + align256(static_cast<int64_t>(D) * D * 2);
    }
    if ((rc = backbone_setup(blocks, n_blocks, D, F, fp8 ? nullptr : pk.data(), pk.data() + n_blocks, pk.data() + 2 * n_blocks,
                             fold_act, qk_norms && rope_cos_sin == nullptr ? norm_product : nullptr, key_lengths, B, T, rows,
                             n_rows, sparse ? hidden_out : nullptr, ffn_split > 1 ? split_counters : qk_counters,
                             ffn_split > 1 ? static_cast<int32_t>(tiles) : (dense_few_rows(M, D, 3 * D, true, false) ? 0 : kQkCounters),
                             as_stream(stream), name)) != TAAC_OK)
      return rc;
  }
  // FP8 mode: scales and e4m3 weights of all blocks (three launches), then the scale of the first block's input
  char* fp8_base = reinterpret_cast<char*>(qk_weight) + align256(static_cast<int64_t>(D) * 4 * n_blocks) +
                   align256(ffn_split_bytes(M, D, F));
  float* fp8_scales = reinterpret_cast<float*>(fp8_base + static_cast<int64_t>(n_blocks) * (fp8 ? fp8_block_bytes(D, F) : 0));
  auto fp8_qkv = [&](int i) { return fp8_base + static_cast<int64_t>(i) * fp8_block_bytes(D, F); };
  auto fp8_out = [&](int i) { return fp8_qkv(i) + align256(static_cast<int64_t>(3) * D * D); };
  auto fp8_ffn = [&](int i) { return fp8_out(i) + align256(static_cast<int64_t>(D) * D); };
  if (fp8 && n_blocks > 0) {
    std::vector<float*> sc(n_blocks);
    std::vector<void*> wq(3 * static_cast<size_t>(n_blocks));
    for (int i = 0; i < n_blocks; ++i) {
      if (blocks[i].query_norm_weight || blocks[i].key_norm_weight)
        return set_error(TAAC_ERR_UNSUPPORTED, "%s: the FP8 mode covers the plain attention layer (no query / key norm)", name);
      if (!blocks[i].attn_norm_weight || !blocks[i].ffn_norm_weight)
        return set_error(TAAC_ERR_INVALID_VALUE, "%s: block %d has a null weight", name, i);
      sc[i] = fp8_scales + 8 * i;
      wq[i] = fp8_qkv(i);
      wq[n_blocks + i] = fp8_out(i);
      wq[2 * n_blocks + i] = fp8_ffn(i);
    }
    if ((rc = fill_zero(fp8_scales, (n_blocks + 1) * 8, as_stream(stream), name)) != TAAC_OK) return rc;
    if ((rc = prepare_backbone_fp8(blocks, n_blocks, D, F, sc.data(), wq.data(), wq.data() + n_blocks,
                                   wq.data() + 2 * n_blocks, as_stream(stream), name)) != TAAC_OK)
      return rc;
    if ((rc = rmsnorm_amax_256(emb, D, blocks[0].attn_norm_weight, eps, M, rows, n_rows, fp8_scales + 4, as_stream(stream),
                               name)) != TAAC_OK)
      return rc;
  }
  // Plain attention layers (no query / key norm, no rotary embedding) with heads of 32 or 64 features keep q | k | v and
  // the attention output as stacks of per-head planes [3 * heads][M][dh] / [heads][M][dh] instead of [M][3 * D] / [M][D]
  // rows: a head's rows are then contiguous for the attention kernel (64-byte pieces of 1 536-byte rows otherwise), and the
  // dense kernels on either side address the planes directly. TAAC_BACKBONE_ROW_MAJOR_QKV keeps the rows (same results).
  const bool planes = fused && !fp8 && !split_out_ffn && (dh == 32 || dh == 64) && !(flags & TAAC_BACKBONE_ROW_MAJOR_QKV);
  const int64_t plane_elems = M * dh;
  const int64_t plane_strides[4] = {static_cast<int64_t>(T) * dh, plane_elems, dh, 1};
  // The last block's kernel (out projection + feed-forward in one) also leaves every token's dot product with the head
  // weight behind, in the q | k | v buffer that is free by then: the readout adds M floats instead of reading the final
  // hidden state again.
  float* token_dots = reinterpret_cast<float*>(qkv);
  const bool head_rides = aligned16(w_head);
  bool dots_ready = false;
  for (int i = 0; i < n_blocks; ++i) {
    const taac_block_weights& w = blocks[i];
    if (!w.attn_norm_weight || !w.qkv_weight || !w.out_weight || !w.ffn_norm_weight || !w.up_weight || !w.down_weight)
      return set_error(TAAC_ERR_INVALID_VALUE, "%s: block %d has a null weight", name, i);
    const bool last = (i == n_blocks - 1);
    const bool ride = last && head_rides;
    bf16_t* x_out = (last && hidden_out != nullptr) ? static_cast<bf16_t*>(hidden_out) : x;
    if (fp8) {
      // Four dense layers with e4m3 operands and per-tensor scales; every activation scale comes out of the epilogue of the
      // kernel that produces the tensor (scales[4..7] = block input, attention output, feed-forward input, hidden state).
      float* sc = fp8_scales + 8 * i;
      PreclearedMaxima precleared;
      if ((rc = taac_norm_linear_fp8_fwd(cur, D, w.attn_norm_weight, eps, fp8_qkv(i), w.qkv_bias, sc + 4, sc + 0, nullptr, 0,
                                         qkv, 3 * D, M, 3 * D, D, rows, n_rows, nullptr, 0.f, nullptr, stream)) != TAAC_OK)
        return rc;
      if ((rc = taac_flash_attn_amax_fwd(qkv, qkv + D, qkv + 2 * D, key_lengths, nullptr, nullptr, nullptr, h, sc + 5, B,
                                         heads, T, T, D / heads, qkv_strides, qkv_strides, qkv_strides, o_strides, 0,
                                         rows ? 2 : 1, TAAC_BF16, stream)) != TAAC_OK)
        return rc;
      if ((rc = taac_norm_linear_fp8_fwd(h, D, nullptr, eps, fp8_out(i), w.out_bias, sc + 5, sc + 1, cur, D, x, D, M, D, D,
                                         rows, n_rows, w.ffn_norm_weight, eps, sc + 6, stream)) != TAAC_OK)
        return rc;
      if ((rc = swiglu_ffn_fp8_readout(x, D, w.ffn_norm_weight, eps, fp8_ffn(i), w.up_bias, w.down_bias, sc + 6, sc + 2, sc + 3,
                                       sc + 7, x, D, x_out, D, M, D, F, 1, rows, n_rows,
                                       last ? nullptr : blocks[i + 1].attn_norm_weight, eps, last ? nullptr : sc + 8 + 4,
                                       ride ? w_head : nullptr, ride ? token_dots : nullptr, stream)) != TAAC_OK)
        return rc;
      dots_ready = ride;
      cur = x_out;
      continue;
    }
    // Fused path: token-stationary kernels with norms and residuals fused, weights repacked into fragment order.
    char* pk_qkv = packed + static_cast<int64_t>(i) * packed_block_bytes(D, F);
    char* pk_out = pk_qkv + align256(static_cast<int64_t>(3) * D * D * 2);
    char* pk_ffn = pk_out + align256(static_cast<int64_t>(D) * D * 2);
    const int ffn_folded = (w.ffn_norm_weight != nullptr ? TAAC_FOLDED_NORM : 0) | (fold_act ? TAAC_FOLDED_ACTIVATION : 0);
    // attention half
    if ((w.query_norm_weight == nullptr) != (w.key_norm_weight == nullptr))
      return set_error(TAAC_ERR_INVALID_VALUE, "%s: block %d: query and key norm weights come together", name, i);
    const bool qk_norm = w.query_norm_weight != nullptr;
    const bool qk_prepare = qk_norm || rope_cos_sin != nullptr;
    const float* q_scale = nullptr;
    const float* k_scale = nullptr;
    const float* q_col_scale = nullptr;
    if (fused && qk_prepare) {
      // The norm statistic comes out of the projection's epilogue and the per-token factor of the norm is applied by
      // the attention kernel. Without a rotation the two norm weights go to the attention kernel as well, as their
      // product on the query features; with one, the epilogue applies weight and rotation. Either way there is no
      // pass of its own over q and k.
      const bool weights_in_epilogue = qk_norm && rope_cos_sin != nullptr;
      if (qk_norm && !weights_in_epilogue) q_col_scale = norm_product + static_cast<int64_t>(i) * D;
      const void* q_weight = weights_in_epilogue ? w.query_norm_weight : nullptr;
      const void* k_weight = weights_in_epilogue ? w.key_norm_weight : nullptr;
      if (weights_in_epilogue && (!planes || !aligned16(q_weight) || !aligned16(k_weight))) {
        if (hipMemcpyAsync(qk_weight, w.query_norm_weight, static_cast<size_t>(D) * 2, hipMemcpyDeviceToDevice,
                           as_stream(stream)) != hipSuccess ||
            hipMemcpyAsync(qk_weight + D, w.key_norm_weight, static_cast<size_t>(D) * 2, hipMemcpyDeviceToDevice,
                           as_stream(stream)) != hipSuccess)
          return set_error(TAAC_ERR_LAUNCH, "%s: copy of the query / key norm weights failed", name);
        q_weight = qk_weight;
        k_weight = qk_weight + D;
      }
      if (planes)
        rc = norm_linear_qk_heads(cur, D, w.attn_norm_weight, eps, w.qkv_bias, pk_qkv, qkv, M, D, heads, T, q_weight,
                                  k_weight, rope_cos_sin, qk_norm ? qk_sumsq : nullptr, qk_norm ? qk_rstd : nullptr, qk_counters, rows,
                                  n_rows, w.attn_norm_weight != nullptr, stream);
      else
        rc = taac_norm_linear_qk_fwd(cur, D, w.attn_norm_weight, eps, nullptr, w.qkv_bias, pk_qkv, qkv, 3 * D, M, D, heads,
                                     T, weights_in_epilogue ? qk_weight : nullptr, rope_cos_sin,
                                     qk_norm ? qk_sumsq : nullptr, rows, n_rows, nullptr, w.attn_norm_weight != nullptr,
                                     stream);
      if (rc != TAAC_OK) return rc;
      if (qk_norm) {
        if (!planes &&
            (rc = taac_row_rstd(qk_sumsq, M, D, eps, qk_rstd, rows, n_rows, stream)) != TAAC_OK)
          return rc;
        q_scale = qk_rstd;
        k_scale = qk_rstd + M;
      }
    } else if (planes) {
      if ((rc = taac_norm_linear_heads_fwd(cur, D, w.attn_norm_weight, eps, w.qkv_bias, pk_qkv, qkv, dh, M, 3 * D, D, rows,
                                           n_rows, w.attn_norm_weight != nullptr, stream)) != TAAC_OK)
        return rc;
    } else if (fused) {
      if ((rc = taac_norm_linear_fwd(cur, D, w.attn_norm_weight, eps, nullptr, w.qkv_bias, pk_qkv, nullptr, 0, qkv,
                                     3 * D, M, 3 * D, D, rows, n_rows, nullptr, w.attn_norm_weight != nullptr,
                                     stream)) != TAAC_OK)
        return rc;
    } else {
      if ((rc = taac_rmsnorm_fwd(cur, w.attn_norm_weight, h, M, D, eps, TAAC_BF16, stream)) != TAAC_OK) return rc;
      if ((rc = taac_linear_bf16(h, D, w.qkv_weight, w.qkv_bias, nullptr, qkv, 3 * D, M, 3 * D, D, TAAC_EPI_NONE, 1,
                                 stream)) != TAAC_OK)
        return rc;
    }
    if (!fused && qk_prepare) {
      if ((rc = taac_qk_norm_rope_fwd(qkv, qkv + D, 3 * D, qkv, qkv + D, 3 * D, M, T, D, heads, w.query_norm_weight,
                                      w.key_norm_weight, eps, rope_cos_sin, nullptr, nullptr, TAAC_BF16, stream)) !=
          TAAC_OK)
        return rc;
    }
    if (planes) {
      if ((rc = taac_flash_attn_scaled_fwd(qkv, qkv + heads * plane_elems, qkv + 2 * heads * plane_elems, key_lengths,
                                           q_scale, k_scale, q_col_scale, h, B, heads, T, T, dh, plane_strides, plane_strides,
                                           plane_strides, plane_strides, 0, rows ? 2 : 1, TAAC_BF16, stream)) != TAAC_OK)
        return rc;
      if ((rc = attn_out_ffn_readout(h, D, dh, w.out_bias, pk_out, cur, D, w.ffn_norm_weight, eps, w.up_bias, w.down_bias,
                                     pk_ffn, x_out, D, M, D, F, rows, n_rows, ffn_folded,
                                     ride ? w_head : nullptr, ride ? token_dots : nullptr, split_scratch, stream)) != TAAC_OK)
        return rc;
      dots_ready = ride;
      cur = x_out;
      continue;
    }
    if ((rc = taac_flash_attn_scaled_fwd(qkv, qkv + D, qkv + 2 * D, key_lengths, q_scale, k_scale, q_col_scale, h, B,
                                         heads, T, T, dh, qkv_strides, qkv_strides, qkv_strides, o_strides, 0, rows ? 2 : 1,
                                         TAAC_BF16, stream)) != TAAC_OK)
      return rc;
    if (fused && !split_out_ffn) {
      // out projection + residual and the whole feed-forward half in one kernel; the stream between them stays on chip
      if ((rc = attn_out_ffn_readout(h, D, 0, w.out_bias, pk_out, cur, D, w.ffn_norm_weight, eps, w.up_bias, w.down_bias,
                                     pk_ffn, x_out, D, M, D, F, rows, n_rows, ffn_folded,
                                     ride ? w_head : nullptr, ride ? token_dots : nullptr, split_scratch, stream)) != TAAC_OK)
        return rc;
      dots_ready = ride;
    } else if (fused) {
      if ((rc = taac_norm_linear_fwd(h, D, nullptr, eps, nullptr, w.out_bias, pk_out, cur, D, x, D, M, D, D, rows,
                                     n_rows, nullptr, 0, stream)) != TAAC_OK)
        return rc;
      // feed-forward half: RMSNorm -> up -> SiLU-gate -> down -> + residual in one kernel
      if ((rc = taac_swiglu_ffn_fwd(x, D, w.ffn_norm_weight, eps, nullptr, w.up_bias, nullptr, w.down_bias, pk_ffn, x,
                                    D, x_out, D, M, D, F, 1, rows, n_rows, ffn_folded, stream)) != TAAC_OK)
        return rc;
    } else {
      if ((rc = taac_linear_bf16(h, D, w.out_weight, w.out_bias, cur, x, D, M, D, D, TAAC_EPI_RESIDUAL, 1, stream)) !=
          TAAC_OK)
        return rc;
      if ((rc = taac_rmsnorm_fwd(x, w.ffn_norm_weight, h, M, D, eps, TAAC_BF16, stream)) != TAAC_OK) return rc;
      if ((rc = taac_linear_bf16(h, D, w.up_weight, w.up_bias, nullptr, g, F, M, 2 * F, D, TAAC_EPI_SWIGLU, 1,
                                 stream)) != TAAC_OK)
        return rc;
      if ((rc = taac_linear_bf16(g, F, w.down_weight, w.down_bias, x, x_out, D, M, D, F, TAAC_EPI_RESIDUAL, 1,
                                 stream)) != TAAC_OK)
        return rc;
    }
    cur = x_out;
  }
  if (n_blocks == 0 && hidden_out != nullptr) {
    if (hipMemcpyAsync(hidden_out, emb, static_cast<size_t>(M) * D * 2, hipMemcpyDeviceToDevice, as_stream(stream)) !=
        hipSuccess)
      return set_error(TAAC_ERR_LAUNCH, "%s: copy of the embeddings failed", name);
  }
  if (dots_ready) {  // the last block's kernel left every token's dot product with the head weight behind
    const int per = kBlock / kWave;
    hipLaunchKernelGGL(token_dots_head_kernel, dim3((B + per - 1) / per), dim3(kBlock), 0, as_stream(stream), token_dots,
                       key_lengths, static_cast<const bf16_t*>(b_head), p, B, T);
    return check_launch(name);
  }
  return taac_masked_mean_head(cur, key_lengths, w_head, b_head, p, B, T, D, stream);
}

extern "C" int taac_front_rows(const int32_t* rows, const int32_t* n_rows, int32_t B, int32_t T, int32_t* front_rows,
                               int32_t* lengths, void* stream) {
  using namespace taac;
  const char* name = "taac_front_rows";
  if (B < 0 || T < 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (static_cast<int64_t>(B) * T > 0x7fffffffLL - B - 1)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: B * T must fit 32-bit row numbers", name);
  if (B == 0) return TAAC_OK;
  if (!rows || !n_rows || !lengths || (T > 0 && !front_rows)) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  const int64_t threads = static_cast<int64_t>(B) * T > B ? static_cast<int64_t>(B) * T : B;
  hipLaunchKernelGGL(front_rows_kernel, dim3(static_cast<uint32_t>((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     as_stream(stream), rows, n_rows, B, T, front_rows, lengths);
  return check_launch(name);
}

extern "C" int taac_mask_front_bits(const uint32_t* struct_bits, int32_t T, const int32_t* rows, int32_t B,
                                    uint32_t* out_bits, void* stream) {
  using namespace taac;
  const char* name = "taac_mask_front_bits";
  if (B < 0 || T < 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions", name);
  if (T > 4096) return set_error(TAAC_ERR_UNSUPPORTED, "%s: at most 4096 tokens per sample", name);
  if (static_cast<int64_t>(B) * T > 0x7fffffffLL - B - 1)
    return set_error(TAAC_ERR_UNSUPPORTED, "%s: B * T must fit 32-bit row numbers", name);
  if (B == 0 || T == 0) return TAAC_OK;
  if (!struct_bits || !rows || !out_bits) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  const int64_t blocks = static_cast<int64_t>(B) * ((T + kFrontRowsPerBlock - 1) / kFrontRowsPerBlock);
  if (blocks > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: too many rows", name);
  hipLaunchKernelGGL(mask_front_bits_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kBlock),
                     kFrontRowsPerBlock * ((T + 31) / 32) * sizeof(uint32_t), as_stream(stream),
                     struct_bits, T, rows, B, out_bits);
  return check_launch(name);
}

namespace taac {
namespace {

// Workspace of taac_stack_fwd for M = B * T rows.
struct StackLayout {
  bf16_t *qkv, *attended;
  float *sumsq, *scales, *products;  // query / key norms: [2 D / 64][M], [2][M], [n_blocks][D]
  uint32_t* counters;                // [kQkCounters]
  int64_t bytes;
};
StackLayout stack_layout(char* base, int64_t M, int32_t D, int32_t n_blocks, bool qk_norm) {
  StackLayout l{};
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    char* here = base + at;
    at += align256(bytes);
    return here;
  };
  l.qkv = reinterpret_cast<bf16_t*>(take(M * 3 * D * 2));
  l.attended = reinterpret_cast<bf16_t*>(take(M * D * 2));
  if (qk_norm) {
    l.sumsq = reinterpret_cast<float*>(take(qk_sums_bytes(M, D)));
    l.counters = reinterpret_cast<uint32_t*>(take(kQkCounters * 4));
    l.scales = reinterpret_cast<float*>(take(2 * M * 4));
    l.products = reinterpret_cast<float*>(take(static_cast<int64_t>(n_blocks) * D * 4));
  }
  l.bytes = at;
  return l;
}

constexpr int kProductBlocks = 16;
struct StackSetup {
  const bf16_t* tokens;
  bf16_t* out;
  const uint8_t* padding;  // [M]
  float* scales;           // [2 M], or null; with the counters
  uint32_t* counters;      // [kQkCounters]
  float* products;         // of blocks first_block .., n_blocks of them
  int64_t M;
  int32_t D, n_blocks;
  const bf16_t* query[kProductBlocks];
  const bf16_t* key[kProductBlocks];
};

// What a stack needs in front of its blocks: the padded rows of the output (they pass through; the blocks write the others), ones in
// the norm factors (rows outside the index are read by nobody, but a lane that holds such a row multiplies by it), zeros in the counters
// and the products of the query and key norm weights.
__global__ __launch_bounds__(kBlock) void stack_setup_kernel(const StackSetup p) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  const int pieces = p.D / 8;
  if (p.tokens != nullptr && i < p.M * pieces) {
    if (p.padding[i / pieces] != 0) reinterpret_cast<bf16x8*>(p.out)[i] = reinterpret_cast<const bf16x8*>(p.tokens)[i];
  }
  if (p.scales != nullptr && i < 2 * p.M) p.scales[i] = 1.f;
  if (p.scales != nullptr && i < kQkCounters) p.counters[i] = 0u;
  if (i < static_cast<int64_t>(p.n_blocks) * p.D) {
    const int block = static_cast<int>(i / p.D), col = static_cast<int>(i % p.D);
    p.products[i] = static_cast<float>(p.query[block][col]) * static_cast<float>(p.key[block][col]);
  }
}

}  // namespace
}  // namespace taac

extern "C" int64_t taac_stack_fwd_bytes(int32_t B, int32_t T, int32_t D, int32_t n_blocks, int qk_norm) {
  if (B <= 0 || T <= 0 || (D != 128 && D != 256) || n_blocks <= 0) return -1;
  return taac::stack_layout(nullptr, static_cast<int64_t>(B) * T, D, n_blocks, qk_norm != 0).bytes;
}

extern "C" int taac_stack_fwd(const void* tokens, const uint8_t* padding, const int32_t* rows, const int32_t* n_rows,
                              const int32_t* front_rows, const int32_t* lengths, const uint32_t* struct_bits,
                              int64_t struct_sample_stride, const taac_block_weights* blocks, int32_t n_blocks, int32_t B, int32_t T,
                              int32_t D, int32_t H, int32_t F, float attn_eps, float ffn_eps, float qk_eps, int norm_folded,
                              void* workspace, int64_t workspace_bytes, void* out, void* stream) {
  using namespace taac;
  const char* name = "taac_stack_fwd";
  if (B <= 0 || T <= 0 || n_blocks <= 0 || H <= 0 || F <= 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: B, T, n_blocks, H and F must be positive", name);
  if ((D != 128 && D != 256) || D % H != 0) return set_error(TAAC_ERR_UNSUPPORTED, "%s: D must be 128 or 256 and H divide it", name);
  if (!tokens || !padding || !rows || !n_rows || !front_rows || !lengths || !struct_bits || !blocks || !out || !workspace)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: null pointer", name);
  if (!aligned16(tokens) || !aligned16(out) || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: tokens and out must be 16-byte, the workspace 256-byte aligned", name);
  if (tokens == out) return set_error(TAAC_ERR_INVALID_VALUE, "%s: out must not be tokens", name);
  const bool qk_norm = blocks[0].query_norm_weight != nullptr;
  for (int i = 0; i < n_blocks; ++i)
    if ((blocks[i].query_norm_weight != nullptr) != qk_norm || (blocks[i].key_norm_weight != nullptr) != qk_norm)
      return set_error(TAAC_ERR_INVALID_VALUE, "%s: query and key norms in all blocks or in none", name);
  const int64_t M = static_cast<int64_t>(B) * T;
  if (M > 0x3fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: at most 2^30 rows", name);
  const StackLayout l = stack_layout(static_cast<char*>(workspace), M, D, n_blocks, qk_norm);
  if (workspace_bytes < l.bytes) return set_error(TAAC_ERR_INVALID_VALUE, "%s: the workspace must hold taac_stack_fwd_bytes", name);
  hipStream_t s = as_stream(stream);
  for (int first = 0; first == 0 || (qk_norm && first < n_blocks); first += kProductBlocks) {
    StackSetup setup{};
    setup.M = M;
    setup.D = D;
    if (first == 0) {
      setup.tokens = static_cast<const bf16_t*>(tokens);
      setup.out = static_cast<bf16_t*>(out);
      setup.padding = padding;
      setup.scales = l.scales;
      setup.counters = l.counters;
    }
    if (qk_norm) {
      setup.products = l.products + static_cast<int64_t>(first) * D;
      setup.n_blocks = n_blocks - first < kProductBlocks ? n_blocks - first : kProductBlocks;
      for (int i = 0; i < setup.n_blocks; ++i) {
        setup.query[i] = static_cast<const bf16_t*>(blocks[first + i].query_norm_weight);
        setup.key[i] = static_cast<const bf16_t*>(blocks[first + i].key_norm_weight);
      }
    }
    const int64_t wide = first == 0 ? std::max<int64_t>(M * (D / 8), kQkCounters) : 0;  // (2 M <= M D / 8)
    const int64_t threads = std::max<int64_t>(wide, static_cast<int64_t>(setup.n_blocks) * D);
    hipLaunchKernelGGL(stack_setup_kernel, dim3(static_cast<uint32_t>((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, setup);
    const int rc = check_launch(name);
    if (rc != TAAC_OK) return rc;
  }
  const int32_t dh = D / H;
  const int64_t qkv_strides[4] = {static_cast<int64_t>(T) * 3 * D, dh, 3 * static_cast<int64_t>(D), 1};
  const int64_t out_strides[4] = {static_cast<int64_t>(T) * D, dh, D, 1};
  for (int i = 0; i < n_blocks; ++i) {
    const taac_block_weights& w = blocks[i];
    const void* x = i == 0 ? tokens : out;
    int rc = qk_norm ? norm_linear_qk_factors(name, x, D, w.attn_norm_weight, attn_eps, w.qkv_bias, w.qkv_weight, l.qkv, 3 * D, M, D, H,
                                              T, qk_eps, l.sumsq, l.scales, l.counters, front_rows, n_rows, rows, 1, stream)
                     : taac_norm_linear_fwd(x, D, w.attn_norm_weight, attn_eps, nullptr, w.qkv_bias, w.qkv_weight, nullptr, 3 * D, l.qkv,
                                            3 * D, M, 3 * D, D, front_rows, n_rows, rows, 1, stream);
    if (rc != TAAC_OK) return rc;
    rc = taac_flash_attn_masked_fwd(l.qkv, l.qkv + D, l.qkv + 2 * D, lengths, struct_bits, struct_sample_stride, nullptr, nullptr, nullptr,
                                    l.scales, qk_norm ? l.scales + M : nullptr, qk_norm ? l.products + static_cast<int64_t>(i) * D : nullptr,
                                    l.attended, B, H, T, T, dh, qkv_strides, qkv_strides, qkv_strides, out_strides, 2, TAAC_BF16, stream);
    if (rc != TAAC_OK) return rc;
    rc = taac_attn_out_ffn_fwd(l.attended, D, w.out_bias, w.out_weight, x, D, w.ffn_norm_weight, ffn_eps, w.up_bias, w.down_bias, w.up_weight,
                               out, D, M, D, F, rows, n_rows, front_rows, norm_folded, stream);
    if (rc != TAAC_OK) return rc;
  }
  return TAAC_OK;
}
