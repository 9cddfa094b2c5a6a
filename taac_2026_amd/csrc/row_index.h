// Valid-row index of a padded batch, one workgroup per (sample, 256 positions): every workgroup forms the prefix sum of the
// samples in front of its own itself (up to B lengths, or B rows of validity words, spread over its threads), so the index takes one
// launch instead of a scan followed by a fill.
#pragma once

#include "common.h"

namespace taac {
namespace {

constexpr int kRowThreads = 256;

// Whether it does: the prefix sums' work grows with the square of the batch, the scan's (length_offsets_kernel: one workgroup, 256
// samples at a time) with the batch, so the line lies where the loads of all workgroups per sample - B x slabs x words of a sample
// (one for lengths) - pass a constant. One launch / scan and fill, us. Lengths: 64 x 512 4.2 / 7.6, 8192 x 512 26 / 42, 16384 x 512
// 81 / 80, 2048 x 2048 15 / 19, 4096 x 2048 33 / 34, 8192 x 2048 90 / 66, 16384 x 32 44 / 71, 32768 x 32 143 / 138. Bits: 64 x 512
// 4.6 / 9.3, 256 x 512 5.8 / 9.6, 1024 x 512 35 / 17, 8192 x 512 2003 / 101, 64 x 2048 11 / 12, 256 x 2048 39 / 19, 16384 x 32 61 / 73.
inline bool row_index_in_one_launch(int64_t B, int64_t T, bool bits) {
  const int64_t slabs = T > kRowThreads ? (T + kRowThreads - 1) / kRowThreads : 1, words = bits ? (T + 31) / 32 : 1;
  return B * slabs * words <= 16384;
}

__device__ __forceinline__ int32_t clamped_length(const int32_t* __restrict__ lengths, int b, int T) {
  const int32_t len = lengths[b];
  return len < 0 ? 0 : (len > T ? T : len);
}

// Set bits among the first T of sample b's validity row.
__device__ __forceinline__ int32_t valid_bit_count(const uint32_t* __restrict__ bits, int b, int T) {
  const int wpr = (T + 31) / 32;
  int32_t n = 0;
  for (int w = 0; w < wpr; ++w) {
    uint32_t word = bits[static_cast<int64_t>(b) * wpr + w];
    if (w == wpr - 1 && T % 32 != 0) word &= (1u << (T % 32)) - 1u;
    n += __popc(word);
  }
  return n;
}

// Sum of the 256 threads' values, in every thread.
__device__ __forceinline__ int32_t workgroup_sum(int32_t v) {
  __shared__ int32_t wave_sums[kRowThreads / kWave];
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  if (threadIdx.x % kWave == 0) wave_sums[threadIdx.x / kWave] = v;
  __syncthreads();
  int32_t s = 0;
#pragma unroll
  for (int w = 0; w < kRowThreads / kWave; ++w) s += wave_sums[w];
  return s;
}

// Rows of workgroup `unit` = sample * slabs + slab, slabs = ceil(T / 256) (at least 1): rows[offset + t] = b * T + t for the valid
// t < lengths[b]; the first slab of a sample also writes its offset, the last sample the total. offsets = rows + B * T.
__device__ __forceinline__ void write_valid_rows(const int32_t* __restrict__ lengths, int B, int T, int unit,
                                                 int32_t* __restrict__ rows, int32_t* __restrict__ n_rows) {
  const int slabs = T > kRowThreads ? (T + kRowThreads - 1) / kRowThreads : 1;
  const int b = unit / slabs, slab = unit % slabs;
  int32_t before = 0;
  for (int i = threadIdx.x; i < b; i += kRowThreads) before += clamped_length(lengths, i, T);
  const int32_t offset = workgroup_sum(before);
  const int32_t len = clamped_length(lengths, b, T);
  const int t = slab * kRowThreads + static_cast<int>(threadIdx.x);
  if (t < len) rows[offset + t] = b * T + t;
  if (slab == 0 && threadIdx.x == 0) {
    int32_t* offsets = rows + static_cast<int64_t>(B) * T;
    offsets[b] = offset;
    if (b == B - 1) {
      offsets[B] = offset + len;
      *n_rows = offset + len;
    }
  }
}

// The same for a validity bit row per sample: token t goes to slot offset + (number of valid tokens of the sample before t).
__device__ __forceinline__ void write_valid_rows_bits(const uint32_t* __restrict__ bits, int B, int T, int unit,
                                                      int32_t* __restrict__ rows, int32_t* __restrict__ n_rows) {
  const int slabs = T > kRowThreads ? (T + kRowThreads - 1) / kRowThreads : 1;
  const int b = unit / slabs, slab = unit % slabs;
  int32_t before = 0;
  for (int i = threadIdx.x; i < b; i += kRowThreads) before += valid_bit_count(bits, i, T);
  const int32_t offset = workgroup_sum(before);
  const int t = slab * kRowThreads + static_cast<int>(threadIdx.x);
  const int wpr = (T + 31) / 32;
  const uint32_t* row = bits + static_cast<int64_t>(b) * wpr;
  if (t < T) {
    const uint32_t word = row[t / 32];
    if ((word >> (t % 32)) & 1u) {
      int32_t rank = __popc(word & ((1u << (t % 32)) - 1u));
      for (int w = 0; w < t / 32; ++w) rank += __popc(row[w]);
      rows[offset + rank] = b * T + t;
    }
  }
  if (slab == 0 && threadIdx.x == 0) {
    int32_t* offsets = rows + static_cast<int64_t>(B) * T;
    offsets[b] = offset;
    if (b == B - 1) {
      const int32_t n = offset + valid_bit_count(bits, b, T);
      offsets[B] = n;
      *n_rows = n;
    }
  }
}

}  // namespace
}  // namespace taac
