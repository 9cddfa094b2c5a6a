// Multi-hot embedding lookup with mean pooling for gfx950: out[b, :] = mean over the non-padding ids of bag b of
// weight[id, :], id 0 = padding, an all-padding bag gives zeros (F.embedding_bag(values, weight, mode="mean",
// padding_idx=0), accelerators/embedding/embedding_bag.py:82-83).
//
// HBM-bound gather: a bag is owned by G consecutive lanes, each holding NV 16-byte pieces of the embedding row, so a
// table row is fetched as one contiguous run of 16-byte requests and the output row is written once. The ids of a bag
// are read four at a time and the (up to four) rows they name are requested before any of them is accumulated, fp32
// accumulation, one rounding.
#include <type_traits>

#include "common.h"

namespace taac {
namespace {

constexpr int kBlock = 256;

template <typename T>
struct Piece;  // one 16-byte piece of a row
template <>
struct Piece<float> {
  static constexpr int N = 4;
  typedef f32x4 vec;
};
template <>
struct Piece<bf16_t> {
  static constexpr int N = 8;
  typedef bf16x8 vec;
};
template <>
struct Piece<f16_t> {
  static constexpr int N = 8;
  typedef f16x8 vec;
};

template <typename T, typename I, int G, int NV>
__global__ __launch_bounds__(kBlock) void embedding_bag_mean_kernel(const T* __restrict__ weight, int64_t num_embeddings,
                                                                     int emb_dim, const I* __restrict__ values,
                                                                     int64_t bags, int bag_size, T* __restrict__ out,
                                                                     int32_t* __restrict__ invalid_count) {
  typedef typename Piece<T>::vec vec_t;
  constexpr int N = Piece<T>::N;
  constexpr int GPB = kBlock / G;
  const int lane = threadIdx.x % G;
  const int64_t bag = static_cast<int64_t>(blockIdx.x) * GPB + threadIdx.x / G;
  if (bag >= bags) return;
  const int nvec = emb_dim / N;
  const I* ids = values + bag * bag_size;
  float acc[NV][N];
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int e = 0; e < N; ++e) acc[i][e] = 0.f;
  int count = 0, invalid = 0;
  for (int j0 = 0; j0 < bag_size; j0 += 4) {
    int64_t id[4];
    bool use[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      id[j] = j0 + j < bag_size ? static_cast<int64_t>(ids[j0 + j]) : 0;
      use[j] = id[j] > 0 && id[j] < num_embeddings;
      invalid += (id[j] < 0 || id[j] >= num_embeddings) ? 1 : 0;
      count += use[j] ? 1 : 0;
    }
    vec_t piece[4][NV];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int v = lane + i * G;
        if (use[j] && v < nvec) piece[j][i] = *reinterpret_cast<const vec_t*>(weight + id[j] * emb_dim + v * N);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int v = lane + i * G;
        if (use[j] && v < nvec) {
#pragma unroll
          for (int e = 0; e < N; ++e) acc[i][e] += static_cast<float>(piece[j][i][e]);
        }
      }
  }
  const float inv = 1.0f / static_cast<float>(count > 0 ? count : 1);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = lane + i * G;
    if (v < nvec) {
      vec_t o;
#pragma unroll
      for (int e = 0; e < N; ++e) o[e] = static_cast<T>(acc[i][e] * inv);
      __builtin_nontemporal_store(o, reinterpret_cast<vec_t*>(out + bag * emb_dim + v * N));
    }
  }
  if (invalid_count != nullptr && lane == 0 && invalid > 0) atomicAdd(invalid_count, invalid);
}

// Rows that are not a whole number of 16-byte pieces, or unaligned tables: one lane per element.
template <typename T, typename I>
__global__ __launch_bounds__(kBlock) void embedding_bag_mean_generic_kernel(const T* __restrict__ weight,
                                                                             int64_t num_embeddings, int emb_dim,
                                                                             const I* __restrict__ values, int64_t bags,
                                                                             int bag_size, T* __restrict__ out,
                                                                             int32_t* __restrict__ invalid_count) {
  const int64_t bag = blockIdx.x;
  const I* ids = values + bag * bag_size;
  for (int c = threadIdx.x; c < emb_dim; c += kBlock) {
    float acc = 0.f;
    int count = 0, invalid = 0;
    for (int j = 0; j < bag_size; ++j) {
      const int64_t id = static_cast<int64_t>(ids[j]);
      if (id > 0 && id < num_embeddings) {
        acc += static_cast<float>(weight[id * emb_dim + c]);
        ++count;
      } else if (id != 0) {
        ++invalid;
      }
    }
    out[bag * emb_dim + c] = static_cast<T>(acc / static_cast<float>(count > 0 ? count : 1));
    if (invalid_count != nullptr && c == 0 && invalid > 0) atomicAdd(invalid_count, invalid);
  }
}

template <typename T, typename I, int G, int NV>
void launch_bag(const T* w, int64_t n, int e, const I* v, int64_t bags, int bag_size, T* out, int32_t* invalid,
                hipStream_t s) {
  constexpr int GPB = kBlock / G;
  hipLaunchKernelGGL((embedding_bag_mean_kernel<T, I, G, NV>), dim3(static_cast<uint32_t>((bags + GPB - 1) / GPB)),
                     dim3(kBlock), 0, s, w, n, e, v, bags, bag_size, out, invalid);
}

template <typename T, typename I>
int dispatch_bag(const void* weight, int64_t n, int e, const void* values, int64_t bags, int bag_size, void* out,
                 int32_t* invalid, hipStream_t s) {
  const T* w = static_cast<const T*>(weight);
  const I* v = static_cast<const I*>(values);
  T* o = static_cast<T*>(out);
  constexpr int N = Piece<T>::N;
  const int nvec = e / N;
  if (e % N != 0 || !aligned16(w) || !aligned16(o) || nvec > 64 * 8) {
    hipLaunchKernelGGL((embedding_bag_mean_generic_kernel<T, I>), dim3(static_cast<uint32_t>(bags)), dim3(kBlock), 0, s, w,
                       n, e, v, bags, bag_size, o, invalid);
    return TAAC_OK;
  }
#define TAAC_BAG_CASE(G, NV)                                          \
  launch_bag<T, I, G, NV>(w, n, e, v, bags, bag_size, o, invalid, s); \
  return TAAC_OK;
  if (nvec <= 1) { TAAC_BAG_CASE(1, 1) }
  if (nvec <= 2) { TAAC_BAG_CASE(2, 1) }
  if (nvec <= 4) { TAAC_BAG_CASE(4, 1) }
  if (nvec <= 8) { TAAC_BAG_CASE(8, 1) }
  if (nvec <= 16) { TAAC_BAG_CASE(16, 1) }
  if (nvec <= 32) { TAAC_BAG_CASE(32, 1) }
  if (nvec <= 64) { TAAC_BAG_CASE(64, 1) }
  if (nvec <= 128) { TAAC_BAG_CASE(64, 2) }
  if (nvec <= 256) { TAAC_BAG_CASE(64, 4) }
  TAAC_BAG_CASE(64, 8)
#undef TAAC_BAG_CASE
}

// Backward of the mean: every valid id j of bag b receives grad_out[b, :] / max(count_b, 1) on row id of the table's
// gradient (accelerators/embedding/kernels/triton.py:105-150, tilelang.py:95-140). The sums are formed in fp32 with
// the hardware's float add-to-memory; rows named by several bags therefore add in an order that varies from launch to
// launch (last-bit differences), as in the reference's atomic adds. One bag per G lanes like the forward; each lane keeps
// its slice of the scaled gradient row in registers over the bag's ids.
template <typename T, typename I>
__global__ __launch_bounds__(kBlock) void embedding_bag_mean_bwd_kernel(const I* __restrict__ values, int64_t bags,
                                                                         int bag_size, const T* __restrict__ grad_out,
                                                                         float* __restrict__ grad_sum,
                                                                         int64_t num_embeddings, int emb_dim, int lanes) {
  const int per_block = kBlock / lanes;
  const int lane = threadIdx.x % lanes;
  const int64_t bag = static_cast<int64_t>(blockIdx.x) * per_block + threadIdx.x / lanes;
  if (bag >= bags) return;
  const I* ids = values + bag * bag_size;
  int count = 0;
  for (int j = 0; j < bag_size; ++j) {
    const int64_t id = static_cast<int64_t>(ids[j]);
    count += (id > 0 && id < num_embeddings) ? 1 : 0;
  }
  if (count == 0) return;
  const float inv = 1.0f / static_cast<float>(count);
  for (int c0 = 0; c0 < emb_dim; c0 += 4 * lanes) {
    float g[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = c0 + e * lanes + lane;
      g[e] = c < emb_dim ? static_cast<float>(grad_out[bag * emb_dim + c]) * inv : 0.f;
    }
    for (int j = 0; j < bag_size; ++j) {
      const int64_t id = static_cast<int64_t>(ids[j]);
      if (id <= 0 || id >= num_embeddings) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = c0 + e * lanes + lane;
        if (c < emb_dim) unsafeAtomicAdd(grad_sum + id * emb_dim + c, g[e]);
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void clear_sums_kernel(float* __restrict__ sums, int64_t count) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
  const int64_t quads = count / 4;
  f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < quads; i += stride)
    reinterpret_cast<f32x4*>(sums)[i] = zero;
  for (int64_t i = quads * 4 + static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < count; i += stride) sums[i] = 0.f;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void round_sums_kernel(const float* __restrict__ sums, T* __restrict__ out,
                                                             int64_t count) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < count; i += stride)
    out[i] = static_cast<T>(sums[i]);
}

template <typename T, typename I>
void launch_bag_bwd(const void* values, int64_t bags, int bag_size, const void* grad_out, float* sums, int64_t n, int e,
                    hipStream_t s) {
  int lanes = 1;
  while (lanes < 64 && lanes * 4 < e) lanes *= 2;
  const int per_block = kBlock / lanes;
  hipLaunchKernelGGL((embedding_bag_mean_bwd_kernel<T, I>), dim3(static_cast<uint32_t>((bags + per_block - 1) / per_block)),
                     dim3(kBlock), 0, s, static_cast<const I*>(values), bags, bag_size, static_cast<const T*>(grad_out),
                     sums, n, e, lanes);
}

// ---- the same gradient without sums in memory -------------------------------------------------------------------------------
// The kernels above add every slot's row to an fp32 copy of the table in memory: the copy is cleared, hit by one atomic per
// slot and feature, and read again to be rounded (1 000 000 x 64 in fp16, 786 000 slots: 37 + 176 + 95 us). Here the slots are
// sorted by the row they name - a count per row, a start per row, the slots placed - and a row's sum is formed in registers and
// written once, rounded. The order within a row, and the order of the rows' segments, is whatever the atomics gave. Rows named
// more than kHot times are cut into chunks that workgroups of their own sum up; the row then adds those.
// The sort is bound by its atomics (one per slot on counts of every row in memory: 57 us of 94 for the above) and its scattered
// accesses. It therefore goes over kBuckets sets of rows: a workgroup counts its share of the slots per set in LDS and reserves
// its places with one add per set, places the slots set by set, and one workgroup per set then counts, scans and places by row
// in LDS. The sets are dealt out in runs of kRun rows, so that popular neighbours spread over all of them, in single rows where the
// table is small enough that its counts stay in L2 (16 000 rows, 262 144 slots under a 1 / id popularity 89 -> 61 us). A set is one
// workgroup's work, however many slots name it: see bag_sort for what that costs. Measured for the
// above: counts 10, places 13, sort 13 us; the whole gradient 145 -> 91 us, 40 000 x 64 with 400 000 x 10 slots 691 -> 216, 2 000 000 x 16
// with 524 288 x 12 528 -> 260. 4096 slots a share: with half as many the adds on the sets' cursors cost more (98 us) than the
// second workgroup per compute unit gives.
// A small table with many slots is counted as a whole in LDS instead, one of very many rows with many slots in memory.
// Bound: the table's gradient (written once) and the gathered rows of grad_out.
constexpr int kHot = 64;        // longest row that one lane group sums by itself
constexpr int kHotChunk = 256;  // entries of a chunk, at least
constexpr int kHotParts = 64;   // chunks of a row, at most
constexpr int kRowsPerThread = 8;
constexpr int kLocalRows = 16384;  // largest table whose counts a workgroup keeps in LDS
constexpr int kLocalThreads = 1024;
constexpr int kBuckets = 256;       // sets of rows
constexpr int kRun = 8;             // consecutive rows of a set; its rows are a multiple of that
constexpr int kBucketRows = kLocalThreads * kRowsPerThread;  // rows of a set that are counted at once
constexpr int kCursors = 64 + kBuckets;  // places of the cursors in front of the counts, whole cache lines
constexpr int kBucketShare = 4096;  // slots of a workgroup, at least
constexpr int kBucketShares = 512;  // workgroups, at most (about)
constexpr int kTogether = 32;       // lanes of a wavefront that name one row and add together, at least

struct BagEntry {
  int32_t bag;
  float inv;  // 1 / number of valid ids of the bag
};
struct HotChunk {
  int32_t first, count, chunks;  // entries; chunks of the row (in its first chunk)
};
struct SortedBags {
  int32_t* cursors;  // entries, chunks; per set its entries (cleared together)
  int32_t* counts;   // [rows], behind the cursors; of a hot row after the start kernel: -1 - its first chunk
  int32_t* start;    // [rows]
  int32_t* rank;     // [slots]: place within the row (whole table in LDS), row within the set
  BagEntry* entries; // [slots]
  BagEntry* by_set;  // [slots]: entries set by set
  int32_t* offsets;  // [shares][kBuckets]: where a share's entries of a set begin, within the set
  HotChunk* chunks;  // [slots / kHot]
  float* partial;    // [slots / kHot][emb_dim]
  int32_t set_rows;  // rows of a set, a multiple of kRun; 0: not sorted by sets, rows in their order
  int32_t run_log2;  // consecutive rows of a set
  int32_t share_bags, shares;
  int64_t bytes;

  // Position of a row in counts and start.
  __device__ __forceinline__ int64_t position(int64_t row) const {
    if (set_rows == 0) return row;
    const uint32_t r = static_cast<uint32_t>(row);  // fewer than 2^30 rows
    return static_cast<int64_t>(set_of(r)) * set_rows + row_in_set(r);
  }
  __device__ __forceinline__ uint32_t set_of(uint32_t row) const { return (row >> run_log2) % kBuckets; }
  __device__ __forceinline__ uint32_t row_in_set(uint32_t row) const {
    return ((row >> run_log2) / kBuckets << run_log2) + (row & ((1u << run_log2) - 1));
  }
};
enum class BagSort { kLocal, kSets, kMemory };
// Where the counts of the rows are formed, by size alone. Gradient in us, ids with u^2 / 1 / id popularity / 30 % of the slots on one id.
// kLocal, the whole table in LDS: every workgroup clears and adds up all rows, but its adds to a popular row meet few others. kSets: the
// workgroup of the set with the popular row sorts all slots that name it.
//   3 rows, 65 536 slots in LDS 32 (u^2), by sets 100; 200 rows, 65 536 33 / 37; 1 024 rows, 65 536 44 / 43 / 39, by sets 41 / 42 / 54;
//   262 144 50 / 68 / 68, 48 / 68 / 119.  4 096 rows: 262 144 73 / 75 / 70, 51 / 63 / 116; 524 288 87 / 96 / 99, 83 / 97 / 206; 786 432
//   95 / 104 / 107, 95 / 126 / 284.  16 000 rows: 262 144 101 / 118 / 109, 47 / 62 / 113; 1 048 576 138 / 156 / 150, 93 / 139 / 344; 2 048 000
//   163 / 185 / 215, 137 / 239 / 712.  The line stands where u^2 gains at most a sixth by sets and one popular row would cost threefold.
// kMemory, a returning add per slot: an id that many slots name queues up there (1 000 000 rows, 1 048 576 slots, 10 % of them on one id: in
// memory 1 003, by sets 181; all of them 9 078, 1 106), but a set of more rows than LDS holds walks its slots again for each kBucketRows of
// them. u^2, in memory / by sets: 10 000 000 rows, 30 000 000 slots 2 480 / 2 250; 50 000 000 rows, 6 291 456 1 499 / 1 436, 30 000 000 3 040 /
// 4 400; 100 000 000 rows, 6 291 456 1 850 / 1 850; 200 000 000 rows, 1 048 576 2 480 / 1 860, 6 291 456 3 260 / 3 700, 30 000 000 5 380 /
// 11 900; 10^9 rows, 1 048 576 9 670 / 9 600, 6 291 456 12 500 / 29 700.
BagSort bag_sort(int64_t n, int64_t slots) {
  if (n <= kLocalThreads || (n <= kLocalRows && slots >= 128 * n)) return BagSort::kLocal;
  const int64_t walks = (n + kBuckets * kBucketRows - 1) / (static_cast<int64_t>(kBuckets) * kBucketRows);
  return slots * walks <= 300000000 ? BagSort::kSets : BagSort::kMemory;
}

SortedBags sorted_layout(char* base, int64_t n, int64_t bags, int bag_size, int emb_dim) {
  SortedBags b{};
  char* at = base;
  auto take = [&](int64_t bytes) {
    char* here = at;
    at += (bytes + 255) & ~static_cast<int64_t>(255);
    return here;
  };
  const int64_t slots = bags * bag_size;
  int64_t rows = n;
  if (bag_sort(n, slots) == BagSort::kSets) {
    b.set_rows = static_cast<int32_t>((n + kRun * kBuckets - 1) / (kRun * kBuckets) * kRun);
    b.run_log2 = n <= kLocalRows ? 0 : 3;
    rows = static_cast<int64_t>(b.set_rows) * kBuckets;
    const int64_t share = std::max<int64_t>(kBucketShare, slots / kBucketShares);
    b.share_bags = static_cast<int32_t>(std::max<int64_t>(1, share / bag_size));
    b.shares = static_cast<int32_t>((bags + b.share_bags - 1) / b.share_bags);
  }
  b.cursors = reinterpret_cast<int32_t*>(take((kCursors + rows) * 4));
  b.counts = b.cursors + kCursors;
  b.start = reinterpret_cast<int32_t*>(take(rows * 4));
  b.rank = reinterpret_cast<int32_t*>(take(slots * 4));
  b.entries = reinterpret_cast<BagEntry*>(take(slots * static_cast<int64_t>(sizeof(BagEntry))));
  if (b.set_rows > 0) {
    b.by_set = reinterpret_cast<BagEntry*>(take(slots * static_cast<int64_t>(sizeof(BagEntry))));
    b.offsets = reinterpret_cast<int32_t*>(take(static_cast<int64_t>(b.shares) * kBuckets * 4));
  }
  b.chunks = reinterpret_cast<HotChunk*>(take(slots / kHot * static_cast<int64_t>(sizeof(HotChunk))));
  b.partial = reinterpret_cast<float*>(take(slots / kHot * emb_dim * 4));
  b.bytes = at - base;
  return b;
}

__global__ __launch_bounds__(kBlock) void bag_clear_kernel(int32_t* __restrict__ counts, int64_t n) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * 4;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (i + e < n) counts[i + e] = 0;
}

// One returning add in memory per slot.
template <typename I>
__global__ __launch_bounds__(kBlock) void bag_count_kernel(const I* __restrict__ values, int64_t slots, int64_t n, SortedBags b) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= slots) return;
  const int64_t id = static_cast<int64_t>(values[i]);
  if (id > 0 && id < n) b.rank[i] = atomicAdd(b.counts + id, 1);
}

// A table small enough that a workgroup counts its share of the slots in LDS and reserves each row's places with one add.
template <typename I>
__global__ __launch_bounds__(kLocalThreads) void bag_count_local_kernel(const I* __restrict__ values, int64_t slots, int32_t n,
                                                                        SortedBags b) {
  extern __shared__ int32_t local[];
  const int64_t per = (slots + gridDim.x - 1) / gridDim.x, begin = per * blockIdx.x, end = begin + per < slots ? begin + per : slots;
  for (int32_t r = threadIdx.x; r < n; r += kLocalThreads) local[r] = 0;
  __syncthreads();
  for (int64_t i = begin + threadIdx.x; i < end; i += kLocalThreads) {
    const int64_t id = static_cast<int64_t>(values[i]);
    if (id > 0 && id < n) b.rank[i] = atomicAdd(local + id, 1);
  }
  __syncthreads();
  for (int32_t r = threadIdx.x; r < n; r += kLocalThreads) {
    const int32_t c = local[r];
    if (c > 0) local[r] = atomicAdd(b.counts + r, c);
  }
  __syncthreads();
  for (int64_t i = begin + threadIdx.x; i < end; i += kLocalThreads) {
    const int64_t id = static_cast<int64_t>(values[i]);
    if (id > 0 && id < n) b.rank[i] += local[id];
  }
}

// Exclusive sum of `mine` over the workgroup's threads; `total`: of all of them. wave_sum: one value per wavefront.
template <int WAVES>
__device__ __forceinline__ int32_t block_scan(int32_t mine, int32_t* wave_sum, int32_t& total) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int32_t upto = mine;
#pragma unroll
  for (int d = 1; d < kWave; d *= 2) {
    const int32_t v = __shfl_up(upto, d);
    if (lane >= d) upto += v;
  }
  if (lane == kWave - 1) wave_sum[wave] = upto;
  __syncthreads();
  int32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const int32_t v = wave_sum[w];
    before += w < wave ? v : 0;
    total += v;
  }
  return before + upto - mine;
}

// A row of `count` entries from `at` on: more than kHot of them are cut into chunks. Returns what counts[] then holds.
__device__ __forceinline__ int32_t row_chunks(const SortedBags& b, int32_t at, int32_t count) {
  if (count <= kHot) return count;
  const int32_t by_parts = (count + kHotParts - 1) / kHotParts, len = by_parts > kHotChunk ? by_parts : kHotChunk;
  const int32_t chunks = (count + len - 1) / len;  // at most count / kHot
  const int32_t first = atomicAdd(b.cursors + 1, chunks);
  for (int32_t k = 0; k < chunks; ++k)
    b.chunks[first + k] = HotChunk{at + k * len, count - k * len < len ? count - k * len : len, chunks};
  return -1 - first;
}

// Starts of the rows' segments: a scan inside the workgroup, one add to the common cursor for all of its rows.
__global__ __launch_bounds__(kBlock) void bag_start_kernel(int64_t n, SortedBags b) {
  __shared__ int32_t wave_sum[kBlock / kWave];
  __shared__ int32_t base;
  const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * kRowsPerThread;
  int32_t c[kRowsPerThread], mine = 0;
#pragma unroll
  for (int e = 0; e < kRowsPerThread; ++e) {
    c[e] = r0 + e < n ? b.counts[r0 + e] : 0;
    mine += c[e];
  }
  int32_t total;
  int32_t at = block_scan<kBlock / kWave>(mine, wave_sum, total);
  if (threadIdx.x == 0) base = total > 0 ? atomicAdd(b.cursors, total) : 0;
  __syncthreads();
  at += base;
#pragma unroll
  for (int e = 0; e < kRowsPerThread; ++e) {
    if (r0 + e >= n) break;
    b.start[r0 + e] = at;
    if (c[e] > kHot) b.counts[r0 + e] = row_chunks(b, at, c[e]);
    at += c[e];
  }
}

// ---- by sets of rows ----
// Entries of every set: a share's are counted in LDS and reserved with one add, whose result is where they begin in the set.
template <typename I>
__global__ __launch_bounds__(kLocalThreads) void bag_set_count_kernel(const I* __restrict__ values, int64_t slots, int bag_size, int64_t n,
                                                                      SortedBags b) {
  __shared__ int32_t count[kBuckets];
  constexpr int kAhead = 4;
  for (int t = threadIdx.x; t < kBuckets; t += kLocalThreads) count[t] = 0;
  __syncthreads();
  const int64_t per = static_cast<int64_t>(b.share_bags) * bag_size, begin = per * blockIdx.x, end = begin + per < slots ? begin + per : slots;
  for (int64_t i = begin + threadIdx.x; i < end; i += kAhead * kLocalThreads) {
    int64_t id[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) id[k] = i + k * kLocalThreads < end ? static_cast<int64_t>(values[i + k * kLocalThreads]) : 0;
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      if (id[k] > 0 && id[k] < n) atomicAdd(count + b.set_of(static_cast<uint32_t>(id[k])), 1);
  }
  __syncthreads();
  for (int t = threadIdx.x; t < kBuckets; t += kLocalThreads) {
    const int32_t c = count[t];
    b.offsets[static_cast<int64_t>(blockIdx.x) * kBuckets + t] = c > 0 ? atomicAdd(b.cursors + 2 + t, c) : 0;
  }
}

// The slots set by set, in the shares of the kernel above; one bag per `lanes` lanes (a power of two up to 64).
template <typename I>
__global__ __launch_bounds__(kLocalThreads) void bag_set_place_kernel(const I* __restrict__ values, int64_t bags, int bag_size, int64_t n,
                                                                      int lanes, SortedBags b) {
  __shared__ int32_t next[kBuckets];
  __shared__ int32_t wave_sum[kLocalThreads / kWave];
  const int t = threadIdx.x;
  int32_t total;
  const int32_t set_begin = block_scan<kLocalThreads / kWave>(t < kBuckets ? b.cursors[2 + t] : 0, wave_sum, total);
  if (t < kBuckets) next[t] = set_begin + b.offsets[static_cast<int64_t>(blockIdx.x) * kBuckets + t];
  __syncthreads();
  const int lane = t % lanes;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * b.share_bags;
  const int64_t last = first + b.share_bags < bags ? first + b.share_bags : bags;
  for (int64_t bag = first + t / lanes; bag < last; bag += kLocalThreads / lanes) {  // whole lane groups
    const I* ids = values + bag * bag_size;
    int count = 0;
    for (int j = lane; j < bag_size; j += lanes) {
      const int64_t id = static_cast<int64_t>(ids[j]);
      count += id > 0 && id < n ? 1 : 0;
    }
    for (int d = lanes / 2; d > 0; d /= 2) count += __shfl_xor(count, d);
    const float inv = 1.0f / static_cast<float>(count > 0 ? count : 1);
    for (int j = lane; j < bag_size; j += lanes) {
      const int64_t id = static_cast<int64_t>(ids[j]);
      if (id > 0 && id < n) {
        const int32_t at = atomicAdd(next + b.set_of(static_cast<uint32_t>(id)), 1);
        b.by_set[at] = BagEntry{static_cast<int32_t>(bag), inv};
        b.rank[at] = static_cast<int32_t>(b.row_in_set(static_cast<uint32_t>(id)));
      }
    }
  }
}

// next[r] += 1 for every lane that takes part; returns its value before. Where a popular row fills the set, the lanes that name it add
// together: as adds to one address they queue up, two clocks each (1 000 000 rows, 1 048 576 slots, half of them on one id: 787 -> 579 us).
template <bool RETURN>
__device__ __forceinline__ int32_t add_row(int32_t* next, uint32_t r, bool takes_part) {
  const uint64_t open = __ballot(takes_part);
  int32_t at = 0;
  if (__popcll(open) >= kTogether) {  // wavefront-uniform, as all of this
    const int lane = threadIdx.x % kWave, first = __ffsll(static_cast<unsigned long long>(open)) - 1;
    const uint32_t row = __builtin_amdgcn_readlane(r, first);
    const uint64_t same = __ballot(r == row);
    if (__popcll(same) >= kTogether) {
      if (lane == first) at = atomicAdd(next + row, __popcll(same));
      if (RETURN) at = __builtin_amdgcn_readlane(at, first) + __popcll(same & ((1ull << lane) - 1));
      takes_part = takes_part && r != row;
    }
  }
  if (takes_part) {
    const int32_t own = atomicAdd(next + r, 1);
    if (RETURN) at = own;
  }
  return at;
}

// One workgroup per set: counts, starts and places of its rows in LDS, kBucketRows of them at a time.
__global__ __launch_bounds__(kLocalThreads) void bag_set_sort_kernel(SortedBags b) {
  __shared__ int32_t next[kBucketRows];
  __shared__ int32_t wave_sum[kLocalThreads / kWave];
  const int t = threadIdx.x, set = blockIdx.x;
  int32_t begin;
  block_scan<kLocalThreads / kWave>(t < set ? b.cursors[2 + t] : 0, wave_sum, begin);  // set < kBuckets <= threads
  const int32_t end = begin + b.cursors[2 + set];
  int32_t at0 = begin;
  for (int32_t r0 = 0; r0 < b.set_rows; r0 += kBucketRows) {
    const int32_t mine0 = t * kRowsPerThread;
    __syncthreads();  // the places and sums of the rows before are done with
#pragma unroll
    for (int e = 0; e < kRowsPerThread; ++e) next[t + e * kLocalThreads] = 0;
    __syncthreads();
    for (int32_t i0 = begin; i0 < end; i0 += kLocalThreads) {  // whole wavefronts
      const uint32_t r = i0 + t < end ? static_cast<uint32_t>(b.rank[i0 + t] - r0) : ~0u;
      add_row<false>(next, r, r < static_cast<uint32_t>(kBucketRows));
    }
    __syncthreads();
    int32_t c[kRowsPerThread], mine = 0, total;
#pragma unroll
    for (int e = 0; e < kRowsPerThread; ++e) {
      c[e] = next[mine0 + e];
      mine += c[e];
    }
    int32_t at = at0 + block_scan<kLocalThreads / kWave>(mine, wave_sum, total);
    if (r0 + mine0 < b.set_rows) {  // kRowsPerThread divides set_rows
      int32_t starts[kRowsPerThread];
#pragma unroll
      for (int e = 0; e < kRowsPerThread; ++e) {
        starts[e] = next[mine0 + e] = at;
        const int32_t entries = c[e];
        c[e] = row_chunks(b, at, entries);
        at += entries;
      }
      const int64_t row = static_cast<int64_t>(set) * b.set_rows + r0 + mine0;
#pragma unroll
      for (int e = 0; e < kRowsPerThread; e += 4) {
        *reinterpret_cast<int4*>(b.start + row + e) = int4{starts[e], starts[e + 1], starts[e + 2], starts[e + 3]};
        *reinterpret_cast<int4*>(b.counts + row + e) = int4{c[e], c[e + 1], c[e + 2], c[e + 3]};
      }
    }
    __syncthreads();
    for (int32_t i0 = begin; i0 < end; i0 += kLocalThreads) {
      const uint32_t r = i0 + t < end ? static_cast<uint32_t>(b.rank[i0 + t] - r0) : ~0u;
      const bool takes_part = r < static_cast<uint32_t>(kBucketRows);
      const int32_t place = add_row<true>(next, r, takes_part);
      if (takes_part) b.entries[place] = b.by_set[i0 + t];
    }
    at0 += total;
  }
}

// One bag per `lanes` lanes (a power of two up to 64).
template <typename I>
__global__ __launch_bounds__(kBlock) void bag_place_kernel(const I* __restrict__ values, int64_t bags, int bag_size, int64_t n,
                                                           int lanes, SortedBags b) {
  const int lane = threadIdx.x % lanes;
  const int64_t bag = static_cast<int64_t>(blockIdx.x) * (kBlock / lanes) + threadIdx.x / lanes;
  if (bag >= bags) return;  // whole lane group
  const I* ids = values + bag * bag_size;
  int count = 0;
  for (int j = lane; j < bag_size; j += lanes) {
    const int64_t id = static_cast<int64_t>(ids[j]);
    count += id > 0 && id < n ? 1 : 0;
  }
  for (int d = lanes / 2; d > 0; d /= 2) count += __shfl_xor(count, d);
  const float inv = 1.0f / static_cast<float>(count > 0 ? count : 1);
  for (int j = lane; j < bag_size; j += lanes) {
    const int64_t id = static_cast<int64_t>(ids[j]);
    if (id > 0 && id < n) b.entries[b.start[id] + b.rank[bag * bag_size + j]] = BagEntry{static_cast<int32_t>(bag), inv};
  }
}

// Adds entries first, first + step, ... (below end) to acc, four in flight.
template <typename T>
__device__ __forceinline__ void add_entries(const BagEntry* entries, const T* __restrict__ grad, int emb_dim, bool live,
                                            int32_t first, int32_t end, int32_t step, float (&acc)[Piece<T>::N]) {
  typedef typename Piece<T>::vec vec_t;
  constexpr int N = Piece<T>::N;
  for (int32_t i = first; i < end; i += 4 * step) {
    BagEntry e[4];
    vec_t g[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool in = i + k * step < end;
      e[k] = entries[in ? i + k * step : i];
      if (!in) e[k].bag = -1;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (live && e[k].bag >= 0) g[k] = *reinterpret_cast<const vec_t*>(grad + static_cast<int64_t>(e[k].bag) * emb_dim);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (live && e[k].bag >= 0) {
#pragma unroll
        for (int c = 0; c < N; ++c) acc[c] = fmaf(static_cast<float>(g[k][c]), e[k].inv, acc[c]);
      }
  }
}

template <typename T, int G>
__global__ __launch_bounds__(kBlock) void bag_hot_kernel(const T* __restrict__ grad_out, int emb_dim, SortedBags b) {
  constexpr int N = Piece<T>::N, GROUPS = kBlock / G;
  __shared__ float red[GROUPS][G * N];
  const int lane = threadIdx.x % G, group = threadIdx.x / G;
  const bool live = lane * N < emb_dim;
  const int32_t n_chunks = b.cursors[1];
  for (int32_t c = blockIdx.x; c < n_chunks; c += gridDim.x) {
    const HotChunk chunk = b.chunks[c];
    float acc[N];
#pragma unroll
    for (int e = 0; e < N; ++e) acc[e] = 0.f;
    add_entries<T>(b.entries, grad_out + lane * N, emb_dim, live, chunk.first + group, chunk.first + chunk.count, GROUPS, acc);
#pragma unroll
    for (int e = 0; e < N; ++e) red[group][lane * N + e] = acc[e];
    __syncthreads();
    for (int col = threadIdx.x; col < emb_dim; col += kBlock) {
      float s = 0.f;
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) s += red[g][col];
      b.partial[static_cast<int64_t>(c) * emb_dim + col] = s;
    }
    __syncthreads();
  }
}

template <typename T, int G>
__global__ __launch_bounds__(kBlock) void bag_rows_kernel(const T* __restrict__ grad_out, T* __restrict__ grad_weight, int64_t n,
                                                          int emb_dim, SortedBags b) {
  typedef typename Piece<T>::vec vec_t;
  constexpr int N = Piece<T>::N;
  const int lane = threadIdx.x % G;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (kBlock / G) + threadIdx.x / G;
  if (row >= n) return;
  const bool live = lane * N < emb_dim;
  const int64_t position = b.position(row);
  const int32_t count = b.counts[position], start = b.start[position];
  float acc[N];
#pragma unroll
  for (int e = 0; e < N; ++e) acc[e] = 0.f;
  if (count >= 0) {
    add_entries<T>(b.entries, grad_out + lane * N, emb_dim, live, start, start + count, 1, acc);
  } else if (live) {
    const int32_t first = -1 - count, chunks = b.chunks[first].chunks;
#pragma unroll 4
    for (int32_t k = 0; k < chunks; ++k) {
      const float* part = b.partial + static_cast<int64_t>(first + k) * emb_dim + lane * N;
#pragma unroll
      for (int e = 0; e < N; ++e) acc[e] += part[e];
    }
  }
  if (!live) return;
  vec_t o;
#pragma unroll
  for (int e = 0; e < N; ++e) o[e] = static_cast<T>(acc[e]);
  __builtin_nontemporal_store(o, reinterpret_cast<vec_t*>(grad_weight + row * emb_dim + lane * N));
}

// Whether the sorted form runs: rows of up to 64 whole pieces, 32-bit positions, and enough work that its six launches (against
// three, or two for fp32) do not decide. Measured back to back, sums in memory / sorted, us, skewed ids, a quarter padding -
// 16-bit: 1 000 000 x 64, 262 144 x 4 slots 316 / 91, 1 024 x 4 slots 154 / 40; 100 000 x 64, 1 024 x 4 24 / 19; 20 000 x 64,
// 256 x 4 11.7 / 18.9; 30 000 x 128, 65 536 x 3 95 / 78; 50 000 x 32, 30 000 x 2 24 / 35; 1 000 x 32, 524 288 x 12 4 384 / 229 (3 053
// with the counts in memory), 1 000 x 16, 65 536 x 4 354 / 48, 1 000 x 64, 4 096 x 4 19 / 33.
// fp32, which the other form sums in place: 1 000 000 x 64, 262 144 x 4 219 / 130, 1 024 x 4 43 / 61; 2 000 000 x 64, 524 288 x 4 420 / 237.
bool sorted_bags(int64_t n, int64_t slots, int emb_dim, int dtype) {
  const int piece = dtype == TAAC_F32 ? 4 : 8;
  if (emb_dim % piece != 0 || emb_dim / piece > kWave || slots <= 0 || n > 0x3fffffffLL || slots > 0x3fffffffLL) return false;
  int lanes = 1;
  while (lanes < emb_dim / piece) lanes *= 2;
  if (n * lanes > 0xffffff00LL) return false;  // threads of a launch over the rows
  const int64_t enough = 1 << 22;
  if (dtype == TAAC_F32) return slots * emb_dim >= enough && 2 * slots >= n;
  return slots * emb_dim >= enough || n * emb_dim >= enough;
}

template <typename T, typename I>
int launch_sorted(const I* values, int64_t bags, int bag_size, const T* grad_out, T* grad_weight, int64_t n, int emb_dim, char* workspace,
                  hipStream_t s, const char* name) {
  const int64_t slots = bags * bag_size;
  const SortedBags b = sorted_layout(workspace, n, bags, bag_size, emb_dim);
  auto blocks = [](int64_t threads) { return dim3(static_cast<uint32_t>((threads + kBlock - 1) / kBlock)); };
  int lanes = 1;
  while (lanes < bag_size && lanes < kWave) lanes *= 2;
  const int64_t cleared = kCursors + (b.set_rows > 0 ? 0 : n);
  hipLaunchKernelGGL(bag_clear_kernel, blocks((cleared + 3) / 4), dim3(kBlock), 0, s, b.cursors, cleared);
  if (b.set_rows > 0) {
    hipLaunchKernelGGL(bag_set_count_kernel<I>, dim3(b.shares), dim3(kLocalThreads), 0, s, values, slots, bag_size, n, b);
    hipLaunchKernelGGL(bag_set_place_kernel<I>, dim3(b.shares), dim3(kLocalThreads), 0, s, values, bags, bag_size, n, lanes, b);
    hipLaunchKernelGGL(bag_set_sort_kernel, dim3(kBuckets), dim3(kLocalThreads), 0, s, b);
  } else if (bag_sort(n, slots) == BagSort::kLocal) {
    const int64_t share = std::max<int64_t>(4 * n, 4 * kLocalThreads);  // slots of a workgroup, so that its counts pay
    auto kernel = bag_count_local_kernel<I>;
    const size_t lds = static_cast<size_t>(n) * 4;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLocalRows * 4) != hipSuccess)
      return set_error(TAAC_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", name, lds);
    const uint32_t grid = static_cast<uint32_t>(std::min<int64_t>(std::max<int64_t>(slots / share, 1), 512));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kLocalThreads), lds, s, values, slots, static_cast<int32_t>(n), b);
  } else {
    hipLaunchKernelGGL(bag_count_kernel<I>, blocks(slots), dim3(kBlock), 0, s, values, slots, n, b);
  }
  if (b.set_rows == 0) {
    hipLaunchKernelGGL(bag_start_kernel, blocks((n + kRowsPerThread - 1) / kRowsPerThread), dim3(kBlock), 0, s, n, b);
    hipLaunchKernelGGL(bag_place_kernel<I>, blocks(bags * lanes), dim3(kBlock), 0, s, values, bags, bag_size, n, lanes, b);
  }
  int rc = check_launch(name);
  if (rc != TAAC_OK) return rc;
  auto go = [&](auto g_tag) {
    constexpr int G = decltype(g_tag)::value;
    const int64_t most = slots / kHot;  // chunks, at most
    if (most > 0)
      hipLaunchKernelGGL((bag_hot_kernel<T, G>), dim3(static_cast<uint32_t>(std::min<int64_t>(most, 2048))), dim3(kBlock), 0, s, grad_out,
                         emb_dim, b);
    hipLaunchKernelGGL((bag_rows_kernel<T, G>), blocks(n * G), dim3(kBlock), 0, s, grad_out, grad_weight, n, emb_dim, b);
    return check_launch(name);
  };
  const int pieces = emb_dim / Piece<T>::N;
  if (pieces <= 1) return go(std::integral_constant<int, 1>{});
  if (pieces <= 2) return go(std::integral_constant<int, 2>{});
  if (pieces <= 4) return go(std::integral_constant<int, 4>{});
  if (pieces <= 8) return go(std::integral_constant<int, 8>{});
  if (pieces <= 16) return go(std::integral_constant<int, 16>{});
  if (pieces <= 32) return go(std::integral_constant<int, 32>{});
  return go(std::integral_constant<int, 64>{});
}

}  // namespace
}  // namespace taac

extern "C" int taac_embedding_bag_mean_fwd(const void* weight, int64_t num_embeddings, int32_t emb_dim,
                                           const void* values, int index_is_int64, int64_t bags, int32_t bag_size,
                                           void* out, int32_t* invalid_count, int dtype, void* stream) {
  using namespace taac;
  const char* name = "taac_embedding_bag_mean_fwd";
  if (num_embeddings <= 0 || emb_dim <= 0 || bags < 0 || bag_size < 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: num_embeddings, emb_dim > 0 and bags, bag_size >= 0 required", name);
  if (bags == 0) return TAAC_OK;
  if (!weight || !out || (bag_size > 0 && !values)) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null tensor pointer", name);
  if (bags > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: more than 2^31-1 bags", name);
  hipStream_t s = as_stream(stream);
  int rc;
#define TAAC_BAG_DTYPE(T)                                                                                             \
  rc = index_is_int64 ? dispatch_bag<T, int64_t>(weight, num_embeddings, emb_dim, values, bags, bag_size, out,        \
                                                 invalid_count, s)                                                     \
                      : dispatch_bag<T, int32_t>(weight, num_embeddings, emb_dim, values, bags, bag_size, out,        \
                                                 invalid_count, s)
  switch (dtype) {
    case TAAC_F32: TAAC_BAG_DTYPE(float); break;
    case TAAC_BF16: TAAC_BAG_DTYPE(bf16_t); break;
    case TAAC_F16: TAAC_BAG_DTYPE(f16_t); break;
    default: return set_error(TAAC_ERR_INVALID_VALUE, "%s: unknown dtype %d", name, dtype);
  }
#undef TAAC_BAG_DTYPE
  if (rc != TAAC_OK) return rc;
  return check_launch(name);
}

extern "C" int taac_embedding_bag_mean_bwd(const void* values, int index_is_int64, int64_t bags, int32_t bag_size,
                                           const void* grad_out, void* grad_weight, int64_t num_embeddings,
                                           int32_t emb_dim, void* workspace, int dtype, void* stream) {
  using namespace taac;
  const char* name = "taac_embedding_bag_mean_bwd";
  if (num_embeddings <= 0 || emb_dim <= 0 || bags < 0 || bag_size < 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: num_embeddings, emb_dim > 0 and bags, bag_size >= 0 required", name);
  if (dtype != TAAC_F32 && dtype != TAAC_BF16 && dtype != TAAC_F16)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: unknown dtype %d", name, dtype);
  if (!grad_weight || (bags > 0 && (!grad_out || (bag_size > 0 && !values))))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: null tensor pointer", name);
  if (dtype != TAAC_F32 && !workspace)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: a 16-bit table gradient needs the fp32 workspace (num_embeddings * emb_dim floats)", name);
  if (bags > 0x7fffffffLL) return set_error(TAAC_ERR_UNSUPPORTED, "%s: more than 2^31-1 bags", name);
  if ((reinterpret_cast<uintptr_t>(dtype == TAAC_F32 ? grad_weight : workspace) & 15) != 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: the fp32 sums must be 16-byte aligned", name);
  hipStream_t s = as_stream(stream);
  float* sums = static_cast<float*>(dtype == TAAC_F32 ? grad_weight : workspace);
  const int64_t count = num_embeddings * emb_dim;
  const uint32_t wide = static_cast<uint32_t>(std::min<int64_t>((count / 4 + kBlock) / kBlock, 256 * 16));
  hipLaunchKernelGGL(clear_sums_kernel, dim3(wide), dim3(kBlock), 0, s, sums, count);
  if (bags > 0 && bag_size > 0) {
#define TAAC_BAG_BWD(T)                                                                                            \
  index_is_int64 ? launch_bag_bwd<T, int64_t>(values, bags, bag_size, grad_out, sums, num_embeddings, emb_dim, s) \
                 : launch_bag_bwd<T, int32_t>(values, bags, bag_size, grad_out, sums, num_embeddings, emb_dim, s)
    if (dtype == TAAC_F32) TAAC_BAG_BWD(float);
    else if (dtype == TAAC_BF16) TAAC_BAG_BWD(bf16_t);
    else TAAC_BAG_BWD(f16_t);
#undef TAAC_BAG_BWD
  }
  if (dtype != TAAC_F32) {
    const uint32_t blocks = static_cast<uint32_t>(std::min<int64_t>((count + kBlock - 1) / kBlock, 256 * 16));
    if (dtype == TAAC_BF16)
      hipLaunchKernelGGL((round_sums_kernel<bf16_t>), dim3(blocks), dim3(kBlock), 0, s, sums, static_cast<bf16_t*>(grad_weight), count);
    else
      hipLaunchKernelGGL((round_sums_kernel<f16_t>), dim3(blocks), dim3(kBlock), 0, s, sums, static_cast<f16_t*>(grad_weight), count);
  }
  return check_launch(name);
}

extern "C" int64_t taac_embedding_bag_mean_bwd_bytes(int64_t num_embeddings, int32_t emb_dim, int64_t bags, int32_t bag_size, int dtype) {
  using namespace taac;
  if (num_embeddings <= 0 || emb_dim <= 0 || bags < 0 || bag_size < 0 || (dtype != TAAC_F32 && dtype != TAAC_BF16 && dtype != TAAC_F16)) return -1;
  const int64_t slots = bags * bag_size;
  if (sorted_bags(num_embeddings, slots, emb_dim, dtype)) return sorted_layout(nullptr, num_embeddings, bags, bag_size, emb_dim).bytes;
  return dtype == TAAC_F32 ? 0 : num_embeddings * emb_dim * 4;
}

extern "C" int taac_embedding_bag_mean_bwd_sized(const void* values, int index_is_int64, int64_t bags, int32_t bag_size,
                                                 const void* grad_out, void* grad_weight, int64_t num_embeddings, int32_t emb_dim,
                                                 void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  using namespace taac;
  const char* name = "taac_embedding_bag_mean_bwd_sized";
  const int64_t need = taac_embedding_bag_mean_bwd_bytes(num_embeddings, emb_dim, bags, bag_size, dtype);
  if (need < 0) return set_error(TAAC_ERR_INVALID_VALUE, "%s: bad dimensions or dtype", name);
  if (workspace_bytes < need || (need > 0 && !workspace))
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: the workspace must hold taac_embedding_bag_mean_bwd_bytes", name);
  const int64_t slots = bags * bag_size;
  if (!sorted_bags(num_embeddings, slots, emb_dim, dtype) || !aligned16(grad_out) || !aligned16(grad_weight)) {
    if (dtype != TAAC_F32 && workspace_bytes < num_embeddings * emb_dim * 4)
      return set_error(TAAC_ERR_UNSUPPORTED, "%s: grad_out and grad_weight must be 16-byte aligned", name);
    return taac_embedding_bag_mean_bwd(values, index_is_int64, bags, bag_size, grad_out, grad_weight, num_embeddings, emb_dim, workspace,
                                       dtype, stream);
  }
  if (!values || !grad_out || !grad_weight) return set_error(TAAC_ERR_INVALID_VALUE, "%s: null tensor pointer", name);
  if ((reinterpret_cast<uintptr_t>(workspace) & 15) != 0)
    return set_error(TAAC_ERR_INVALID_VALUE, "%s: the workspace must be 16-byte aligned", name);
  hipStream_t s = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
#define TAAC_BAG_SORTED(T)                                                                                                        \
  (index_is_int64 ? launch_sorted<T, int64_t>(static_cast<const int64_t*>(values), bags, bag_size, static_cast<const T*>(grad_out), \
                                              static_cast<T*>(grad_weight), num_embeddings, emb_dim, ws, s, name)                 \
                  : launch_sorted<T, int32_t>(static_cast<const int32_t*>(values), bags, bag_size, static_cast<const T*>(grad_out), \
                                              static_cast<T*>(grad_weight), num_embeddings, emb_dim, ws, s, name))
  if (dtype == TAAC_F32) return TAAC_BAG_SORTED(float);
  if (dtype == TAAC_BF16) return TAAC_BAG_SORTED(bf16_t);
  return TAAC_BAG_SORTED(f16_t);
#undef TAAC_BAG_SORTED
}
