// Receive side: merge many (index, value) payloads.  The reference builds a
// dense zero tensor of the full gradient length, scatter-adds every payload
// into it and extracts the nonzeros again (comm.py:32-50).  Here the entries
// are stably sorted by index, equal indices are summed in fp32 in arrival order
// (the order a sequential scatter_add_ uses, so the result is reproducible),
// zero sums are dropped and the survivors leave in ascending index order.
#include "zen_common.h"
#include "zen_slab.h"
#include "zen_slab_feed.h"
#include "zen_wide.h"

namespace zen {

namespace {

constexpr int kMrgBlock = 512;
constexpr int kMrgItems = 16;  // consecutive sorted entries per thread (few, large tiles: short prefix chain)
constexpr int kMrgTile = kMrgBlock * kMrgItems;

// Validated sort keys.  The payload that travels with a key is the value itself
// (as fp32 bits): the stable sort keeps arrival order, and the reduce kernel
// needs no gather.
template <typename I, typename S>
__global__ __launch_bounds__(256) void k_merge_prep(const I *__restrict__ idx, const S *__restrict__ val, uint32_t r,
                                                    uint32_t dense_n, uint32_t *__restrict__ keys,
                                                    uint32_t *__restrict__ perm, int32_t *status) {
  const uint32_t j = blockIdx.x * 256u + threadIdx.x;
  if (j >= r) return;
  const I k = idx[j];
  const bool ok = k >= 0 && (uint64_t)k < (uint64_t)dense_n;
  if (!ok) atomicOr(status, ZEN_STAT_BAD_INDEX);
  const uint32_t key = ok ? (uint32_t)k : dense_n;  // bad indices sort behind every good one
  keys[j] = key;
  perm[j] = __float_as_uint(KeyOf<S>::to_f32(val[j]));
}

// One tile = kMrgTile consecutive sorted entries.  The tile's keys and values
// are first brought into LDS with coalesced loads; each thread then walks
// kMrgItems consecutive entries in LDS.  A run that continues past the tile is finished from global
// memory by the thread that owns its head.
__device__ inline int mrg_slot(int i) { return i + (i >> 4); }  // one pad word per 16: conflict-free strides

template <typename I, typename O>
__global__ __launch_bounds__(kMrgBlock) void k_merge_reduce(
    const uint32_t *__restrict__ keys, const uint32_t *__restrict__ perm, uint32_t r,
    uint32_t dense_n, I *__restrict__ out_idx, O *__restrict__ out_val, int64_t capacity,
    ScanState st, int ntiles, int64_t *out_count, int32_t *status) {
  __shared__ uint32_t s_scan[kMrgBlock / 64 + 1];
  __shared__ uint64_t s_bcast;
  __shared__ int s_tile;
  __shared__ uint32_t s_key[kMrgTile + kMrgTile / 16];
  __shared__ float s_val[kMrgTile + kMrgTile / 16];
  if (threadIdx.x == 0) s_tile = (int)atomicAdd(st.ticket, 1u);
  __syncthreads();
  const int tile = s_tile;
  if (tile >= ntiles) return;
  const uint32_t tile_base = (uint32_t)tile * kMrgTile;
#pragma unroll
  for (int q = 0; q < kMrgItems; ++q) {
    const int local = q * kMrgBlock + threadIdx.x;
    const uint32_t i = tile_base + local;
    uint32_t k = 0xffffffffu;
    float v = 0.0f;
    if (i < r) {
      k = keys[i];
      v = __uint_as_float(perm[i]);
    }
    s_key[mrg_slot(local)] = k;
    s_val[mrg_slot(local)] = v;
  }
  __syncthreads();
  const int first = threadIdx.x * kMrgItems;
  uint32_t k[kMrgItems];
  float sum[kMrgItems];
  uint32_t keep = 0;
  uint32_t prev = first > 0 ? s_key[mrg_slot(first - 1)] : (tile_base > 0 ? keys[tile_base - 1] : 0xffffffffu);
#pragma unroll
  for (int q = 0; q < kMrgItems; ++q) {
    const int local = first + q;
    k[q] = s_key[mrg_slot(local)];
    const bool head = k[q] < dense_n && ((tile_base + local) == 0 || k[q] != prev);
    prev = k[q];
    sum[q] = 0.0f;
    if (head) {
      float acc = 0.0f;  // the dense tensor starts at +0 (comm.py:35)
      int u = local;
      while (u < kMrgTile && s_key[mrg_slot(u)] == k[q]) acc += s_val[mrg_slot(u++)];
      if (u == kMrgTile)
        for (uint32_t g = tile_base + kMrgTile; g < r && keys[g] == k[q]; ++g)
          acc += __uint_as_float(perm[g]);
      sum[q] = acc;
      if (SumAs<O>::kept(acc)) keep |= 1u << q;
    }
  }
  uint32_t total;
  const uint32_t before = block_exclusive_scan<uint32_t, kMrgBlock>((uint32_t)__popc(keep), s_scan, &total);
  const uint64_t tile_start = lookback_exclusive(st, tile, total, status, &s_bcast);
  if (tile == ntiles - 1 && threadIdx.x == 0) {
    const uint64_t all = tile_start + total;
    *out_count = (int64_t)all;
    if (all > (uint64_t)capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  }
  // compact the kept entries in LDS (everybody is past reading the staged tile:
  // the scan above synchronised), then write them out with consecutive lanes
  uint32_t li = before;
#pragma unroll
  for (int q = 0; q < kMrgItems; ++q) {
    if (keep & (1u << q)) {
      s_key[li] = k[q];
      s_val[li] = sum[q];
      ++li;
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kMrgBlock) {
    const uint64_t pos = tile_start + i;
    if (pos < (uint64_t)capacity) {
      out_idx[pos] = (I)s_key[i];
      out_val[pos] = SumAs<O>::of(s_val[i]);
    }
  }
}

template <typename S>
__global__ __launch_bounds__(256) void k_scatter_dense(const int32_t *__restrict__ idx, const float *__restrict__ sum,
                                                       const int64_t *count, S *__restrict__ dense, uint32_t dense_n);
// The merged indices come out of workspace memory: after a merge that gave up (ZEN_STAT_INTERNAL, ZEN_STAT_RETRY)
// some of them may never have been written, so none is trusted as an address without a look.
template <>
__global__ __launch_bounds__(256) void k_scatter_dense<uint32_t>(const int32_t *__restrict__ idx,
                                                                 const float *__restrict__ sum,
                                                                 const int64_t *count, uint32_t *__restrict__ dense,
                                                                 uint32_t dense_n) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i < *count && (uint32_t)idx[i] < dense_n) dense[idx[i]] = __float_as_uint(sum[i]);
}
template <>
__global__ __launch_bounds__(256) void k_scatter_dense<uint16_t>(const int32_t *__restrict__ idx,
                                                                 const float *__restrict__ sum,
                                                                 const int64_t *count, uint16_t *__restrict__ dense,
                                                                 uint32_t dense_n) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i < *count && (uint32_t)idx[i] < dense_n) dense[idx[i]] = f32_to_bf16_rne(sum[i]);
}

// ---------------------------------------------------------- merge on bucket slabs
//
// The indices a destination receives were assigned to it by a hash, so they spread evenly over [0, dense_n):
// the entries go to bucket slabs by index range (zen_slab_feed.h) as (index, arrival number, value) records,
// and one workgroup per bucket sorts its slab by (index, arrival number) inside LDS (one word per record), sums every run of equal
// indices in arrival order, drops zero sums and writes what is left at the place the buckets before it
// leave off (every bucket publishes how much it keeps and adds up what the earlier ones published).

constexpr int kMergeTarget = 3072;   // records a bucket is sized for: duplicates make the buckets less even
// Twice the threads of the scatter kernels, half the records each: the kernel's phases are chains of LDS round
// trips, which eight waves per SIMD hide better than four, and a thread's records then fit 64 registers, so
// that two workgroups share a compute unit.
constexpr int kMergeBlock = 1024;
constexpr int kMergeRecs = kSlabCap / kMergeBlock;  // slab records per thread
constexpr int kMergeItems = 7;       // sorted records per thread while summing (odd: no LDS bank conflicts)
static_assert(kMergeBlock * kMergeItems >= kSlabCap, "every sorted place needs an owner");

// An entry travels as (index, arrival number, value bits); in the bucket slabs the three sit in arrays of their
// own (the value in its own type: ten bytes per bf16 entry).
template <typename I, typename S>
struct MergeSrc {
  SlabGeom geo;
  const I *idx;
  const S *val;
  uint32_t dense_n;
  int32_t *status;
  // the value is fetched again by arrival number when the entry is written: a workgroup's 4096 arrival numbers
  // are consecutive, so those loads hit the 8 KB it has just read
  using Last = S;
  static constexpr int kStaged = 2;
  __device__ inline uint32_t late(const uint32_t (&w)[3], int) const { return (uint32_t)val[w[1]]; }
  using Raw = I;
  __device__ inline I fetch(uint32_t e) const { return idx[e]; }
  __device__ inline bool load(I k, uint32_t e, uint32_t (&w)[3], uint32_t *bucket) const {
    if (k < 0 || (uint64_t)k >= (uint64_t)dense_n) {
      atomicOr(status, ZEN_STAT_BAD_INDEX);  // skipped, like everything behind the good ones in the general path
      return false;
    }
    w[0] = (uint32_t)k;
    w[1] = e;
    w[2] = 0;
    *bucket = geo.bucket_of((uint32_t)k);
    return true;
  }
};
template <typename S>
struct MergeSink {
  SlabGeom geo;
  uint32_t *slab_idx, *slab_arr;
  S *slab_val;
  __device__ inline bool keep(const uint32_t (&)[3]) const { return true; }
  __device__ inline uint32_t bucket(const uint32_t (&w)[3]) const { return geo.bucket_of(w[0]); }
  __device__ inline void store(size_t at, const uint32_t (&w)[3]) const {
    slab_idx[at] = w[0];
    slab_arr[at] = w[1];
    slab_val[at] = (S)w[2];
  }
};

// The sums of a workgroup's n sorted records (indices in sh.key, value bits in sh.tie), in registers: record q of a thread
// ends a run of equal indices, whose sum is kept, where bit q of the answer is set.  Thread t owns the sorted places
// [t * per, (t + 1) * per), per <= ITEMS odd, which keeps the lanes of a wave on different LDS banks.
template <typename O, typename Shared, int ITEMS>
__device__ inline uint32_t sum_runs(const Shared &sh, uint32_t n, uint32_t per, uint32_t (&k)[ITEMS], float (&sum)[ITEMS]) {
  // It fetches them all at once (also what lies behind the last one, up to kSlabPad words past the slab, which counts for
  // nothing) and walks through them in registers.  A run of equal indices is summed in arrival order from +0 (like the dense
  // tensor of comm.py:35) and belongs to the thread that holds its last record; where that run began before
  // the thread's first place (rare: runs are short next to `per`, long ones come from payloads that overlap),
  // the part in front is summed first, from the run's head on.
  static_assert(ITEMS <= kSlabPad, "words behind the records");
  constexpr uint32_t kNoKey = 0xffffffffu;  // offsets are below the bucket width
  const uint32_t first = threadIdx.x * per;
  const uint32_t left = first < n ? n - first : 0u;
  const uint32_t own = left < per ? left : per;
  const uint32_t from = first < (uint32_t)kSlabCap ? first : (uint32_t)kSlabCap;
  float v[ITEMS];
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    k[q] = sh.key[from + q];
    v[q] = __uint_as_float(sh.tie[from + q]);
  }
  const uint32_t before = sh.key[from > 0 ? from - 1u : 0u], after = sh.key[first + per < n ? first + per : 0u];
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) k[q] = (uint32_t)q < own ? k[q] : kNoKey;
  const uint32_t before_k = first > 0 ? before : kNoKey;
  const uint32_t after_k = first + per < n ? after : kNoKey;
  float acc = 0.0f;
  if (own && before_k == k[0] && after_k != before_k) {
    // the run began before this thread's places and ends here: find its head, sum up to the place in front of `first`
    acc = sum_run_before(sh.key, sh.tie, first, before_k);
  }
  uint32_t keep = 0;
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    const uint32_t prev = q > 0 ? k[q > 0 ? q - 1 : 0] : before_k;
    const uint32_t next = q + 1 < ITEMS ? ((uint32_t)(q + 1) < per ? k[q + 1 < ITEMS ? q + 1 : q] : after_k) : after_k;
    acc = (k[q] != prev ? 0.0f : acc) + v[q];
    sum[q] = acc;
    keep |= (((uint32_t)q < own) & (k[q] != next) & SumAs<O>::kept(acc)) ? 1u << q : 0u;
  }
  return keep;
}

// The first rows of a slab, loaded beside the number of its records (what lies behind the last one is read and not looked
// at: the slab's memory is there), in no branch, so that all loads are in flight together.
constexpr int kMergeAhead = 4;
struct MergeAhead {
  uint32_t idx[kMergeAhead], arr[kMergeAhead];
};

// A bucket's slab (`idx`, `arr`, `val`: n_raw records; indices from `lo` on): sorted, summed, and what is kept put side by
// side to sh.key / sh.tie (visible behind a barrier).  Returns how many entries that are; false in *ranked if the indices
// pile up.  ROWS records of a thread before the sort, ITEMS after it: written out for the numbers that occur, since what
// bounds the kernel is vector instructions (with six rows and seven places for every bucket, addresses of 64 bits for every
// access and counters in an order that took five instructions to find, 318 for every 64 records, 174 so): 6.2 M bf16 entries
// of sixteen lists 74 -> 64 us, 10.7 M fp32 entries beside the encode's kernels 149 -> 137.
template <typename S, typename O, int ROWS, int ITEMS>
__device__ __forceinline__ uint32_t merge_rows(SlabSortShared &sh, const SlabGeom &geo, int tie_bits,
                                               const MergeAhead &ahead, const uint32_t *__restrict__ idx,
                                               const uint32_t *__restrict__ arr, const S *__restrict__ val, uint32_t n_raw,
                                               uint32_t lo, bool *ranked) {
  static_assert(kMergeBlock * ROWS <= kSlabCap && ITEMS % 2 == 1 && ROWS <= ITEMS, "the slab is there, every sorted place has an owner");
  uint32_t off[ROWS], tie[ROWS], rank[ROWS];
  uint32_t live = 0;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const uint32_t j = threadIdx.x + i * kMergeBlock;
    off[i] = i < kMergeAhead ? ahead.idx[i < kMergeAhead ? i : 0] : idx[j];
    tie[i] = i < kMergeAhead ? ahead.arr[i < kMergeAhead ? i : 0] : arr[j];
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    off[i] -= lo;
    live |= (threadIdx.x + i * kMergeBlock < n_raw ? 1u : 0u) << i;
  }
  uint32_t n = 0;
  *ranked = slab_rank<kMergeBlock>(sh, geo, tie_bits, off, tie, live, rank, &n);
  if (!*ranked) return 0;
  // the values only now: kept across the ranking they cost registers that two workgroups a compute unit do not
  // have (6.2 M records: 67 us instead of 64)
  S v[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) v[i] = val[threadIdx.x + i * kMergeBlock];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    if (live & (1u << i)) {
      sh.key[rank[i]] = off[i];
      sh.tie[rank[i]] = __float_as_uint(KeyOf<S>::to_f32(v[i]));  // the arrival numbers have done their work: their place takes the values
    }
  }
  __syncthreads();
  uint32_t k[ITEMS];
  float sum[ITEMS];
  const uint32_t keep = sum_runs<O>(sh, n, (uint32_t)ITEMS, k, sum);
  uint32_t total;
  uint32_t at = block_exclusive_scan<uint32_t, kMergeBlock>((uint32_t)__popc(keep), sh.scan, &total);
  // everybody is past reading the sorted bucket: the scan synchronised
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    if (keep & (1u << q)) {
      sh.key[at] = k[q] + lo;
      sh.tie[at] = __float_as_uint(sum[q]);
      ++at;
    }
  }
  return total;
}

template <typename I, typename S, typename O>
__global__ __launch_bounds__(kMergeBlock, 8) void k_merge_bucket(SlabGeom geo, uint32_t *__restrict__ cursor,
                                                             uint32_t *__restrict__ coarse_cursor,
                                                             const uint32_t *__restrict__ bucket_lo,
                                                             const uint32_t *__restrict__ slab_idx,
                                                             const uint32_t *__restrict__ slab_arr,
                                                             const S *__restrict__ slab_val,
                                                             I *__restrict__ out_idx, O *__restrict__ out_val,
                                                             int64_t capacity, ScanState st, uint32_t *done, int tie_bits,
                                                             int64_t *out_count, HostAnswer answer, int32_t *status) {
  __shared__ SlabSortShared sh;  // the values take the counters' place once the ranks are known
  __shared__ int s_tile;
  if (threadIdx.x == 0) s_tile = (int)atomicAdd(st.ticket, 1u);
  __syncthreads();
  const int b = __builtin_amdgcn_readfirstlane(s_tile);  // buckets are taken in order, so every earlier bucket already runs
  const int nb = (int)geo.nbuckets;
  if (b >= nb) return;
  const size_t base = (size_t)b * kSlabCap;
  const uint32_t *idx = slab_idx + base, *arr = slab_arr + base;
  const S *val = slab_val + base;
  uint32_t n_raw = cursor[b];
  const uint32_t lo = bucket_lo[b];
  MergeAhead ahead;
#pragma unroll
  for (int i = 0; i < kMergeAhead; ++i) {
    ahead.idx[i] = idx[threadIdx.x + i * kMergeBlock];
    ahead.arr[i] = arr[threadIdx.x + i * kMergeBlock];
  }
  if (n_raw > (uint32_t)kSlabCap) n_raw = kSlabCap;  // the scatter flagged the overflow
  // The counters of the scatter kernels go back to zero (this workgroup was the only reader of its slab's
  // count; the coarse cursors a slice per workgroup), and the last workgroup to finish clears the prefix
  // state: the memory that must be zero when a call starts is zero again when it ends.
  for (uint32_t i = (uint32_t)b * kMergeBlock + threadIdx.x; i < kCoarseCursorWords; i += (uint32_t)nb * kMergeBlock)
    coarse_cursor[i] = 0;
  bool ranked;
  uint32_t total;
  if (n_raw <= 3u * kMergeBlock)
    total = merge_rows<S, O, 3, 3>(sh, geo, tie_bits, ahead, idx, arr, val, n_raw, lo, &ranked);
  else if (n_raw <= 4u * kMergeBlock)
    total = merge_rows<S, O, 4, 5>(sh, geo, tie_bits, ahead, idx, arr, val, n_raw, lo, &ranked);
  else if (n_raw <= 5u * kMergeBlock)
    total = merge_rows<S, O, 5, 5>(sh, geo, tie_bits, ahead, idx, arr, val, n_raw, lo, &ranked);
  else
    total = merge_rows<S, O, kMergeRecs, kMergeItems>(sh, geo, tie_bits, ahead, idx, arr, val, n_raw, lo, &ranked);
  if (threadIdx.x == 0) {
    // where the next bucket's output starts: the sum of what all earlier buckets keep.  A bucket that was not ranked
    // contributes nothing; the prefix protocol still gets its (empty) tile
    desc_store(&st.desc[b], kDescAggregate | total);
    cursor[b] = 0;  // every thread has read it: slab_rank synchronised
    if (!ranked) atomicOr(status, ZEN_STAT_RETRY);
  }
  // Every thread asks for a few of the earlier buckets' counts (bounded wait), nobody waits for a chain of prefixes.
  constexpr int kAsk = kSlabMaxBuckets / kMergeBlock;
  uint64_t d[kAsk];
#pragma unroll
  for (int e = 0; e < kAsk; ++e) {
    const int p = (int)threadIdx.x + e * kMergeBlock;
    d[e] = kDescAggregate;
    if (e * kMergeBlock < b && p < b) d[e] = desc_load(&st.desc[p]);
  }
  uint32_t mine = 0;  // (fewer than 2^31 entries in all)
  bool gave_up = false;
#pragma unroll
  for (int e = 0; e < kAsk; ++e) {
    if (e * kMergeBlock >= b) break;
    const int p = (int)threadIdx.x + e * kMergeBlock;
    uint32_t spins = 0;
    while ((d[e] >> 62) == 0) {
      if (++spins > kSpinLimit) {
        gave_up = true;
        break;
      }
      __builtin_amdgcn_s_sleep(2);
      d[e] = desc_load(&st.desc[p]);
    }
    mine += (uint32_t)d[e];
  }
  if (gave_up) atomicOr(status, ZEN_STAT_INTERNAL);
  uint32_t tile_start;
  block_exclusive_scan<uint32_t, kMergeBlock>(mine, sh.scan, &tile_start);  // its barriers also publish the gathered entries
  if (b == nb - 1 && threadIdx.x == 0) {
    const uint64_t all = (uint64_t)tile_start + total;
    // (for the launch's last workgroup to read, on another die maybe)
    __hip_atomic_store(out_count, (int64_t)all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (all > (uint64_t)capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  }
  const uint64_t room = (uint64_t)capacity > tile_start ? (uint64_t)capacity - tile_start : 0;
  const uint32_t fits = total < room ? total : (uint32_t)room;
  I *const to_idx = out_idx + tile_start;
  O *const to_val = out_val + tile_start;
  for (uint32_t i = threadIdx.x; i < fits; i += kMergeBlock) {
    to_idx[i] = (I)sh.key[i];
    to_val[i] = SumAs<O>::of(__uint_as_float(sh.tie[i]));
  }
  // every workgroup has read the descriptors it needs before it gets here
  if (answer.host) wait_global_acks();  // its share of the status word, and the count
  __syncthreads();
  if (threadIdx.x == 0) s_tile = done_last(done, (uint32_t)b, (uint32_t)nb);
  __syncthreads();
  if (s_tile) {
    for (int i = threadIdx.x; i < nb; i += kMergeBlock) st.desc[i] = 0ull;
    for (uint32_t i = threadIdx.x; i < kDoneWords; i += kMergeBlock) done[i] = 0;
    if (threadIdx.x == 0) *st.ticket = 0;
    host_answer_count(answer, out_count, status);
  }
}

// A short list in one workgroup, straight from where it lies: no slabs, no zeroed memory, any indices.  DENSE: out_val is
// the dense tensor, written whole.  Bound by the chain of its phases, LDS round trips and three trips to memory: a rounded
// merge of 1000 entries spread over the range 27 us a call (38 on the tables of the wide buckets, which are laid out for
// 16 384).  Indices that pile up in few of the narrow ranges would be compared pair by pair, some 8000 pairs a microsecond:
// beyond kMergeOnePairs for every entry a compare-exchange network sorts them, which takes about as long as that many
// (6144 entries in a 4096th of a range of 2^30, a call: 2020 us and now 99; 1000 of them 73 and 42).
constexpr uint32_t kMergeOnePairs = 64;
struct MergeOneShared : SlabSortShared {
  static constexpr bool kPairs = true;
  uint32_t pairs, pairs_most;
};
static_assert(offsetof(SlabSortShared, scan) >= kSlabCap * sizeof(uint64_t), "an index and an arrival number for every entry");
constexpr int kMergeOneArrBits = 13;
static_assert(kSlabCap <= (1 << kMergeOneArrBits), "an arrival number");

template <typename I, typename S, typename O, bool DENSE>
__global__ __launch_bounds__(kMergeBlock) void k_merge_one(SlabGeom geo, const void *__restrict__ idx, int idx64,
                                                           const S *__restrict__ val, uint32_t r, uint32_t dense_n,
                                                           I *__restrict__ out_idx, O *__restrict__ out_val, int64_t capacity,
                                                           int tie_bits, int64_t *out_count, HostAnswer answer, int32_t *status) {
  __shared__ union {
    MergeOneShared sh;
    uint64_t both[kSlabCap];  // in the place of the keys and ties
  } s_all;
  MergeOneShared &sh = s_all.sh;
  if (threadIdx.x == 0) sh.pairs_most = kMergeOnePairs * r;
  uint32_t off[kMergeRecs], arr[kMergeRecs], rank[kMergeRecs];
  S v[kMergeRecs];
  uint32_t live = 0;
  {
    int64_t at[kMergeRecs];
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i) {
      const uint32_t j = threadIdx.x + i * kMergeBlock;
      at[i] = 0;
      v[i] = 0;
      if ((uint32_t)(i * kMergeBlock) >= r) continue;  // the same for the whole workgroup
      const uint32_t e = j < r ? j : 0u;
      at[i] = idx64 ? static_cast<const int64_t *>(idx)[e] : (int64_t)static_cast<const int32_t *>(idx)[e];
      v[i] = val[e];
    }
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i) {
      const uint32_t j = threadIdx.x + i * kMergeBlock;
      const bool good = at[i] >= 0 && at[i] < (int64_t)dense_n;
      off[i] = good ? (uint32_t)at[i] : 0u;
      arr[i] = j;
      if (j < r && good) live |= 1u << i;
      bad |= j < r && !good;
    }
    if (bad) atomicOr(status, ZEN_STAT_BAD_INDEX);  // skipped
  }
  if (DENSE) {  // zeros, while the records are ranked
    constexpr uint32_t V = 16 / sizeof(O);
    const uint32_t skew = (uint32_t)((reinterpret_cast<uintptr_t>(out_val) & 15u) / sizeof(O));
    uint32_t head = (V - skew) % V;
    if (head > dense_n) head = dense_n;
    const uint32_t vecs = (dense_n - head) / V;
    const u32x4 zero = {0, 0, 0, 0};
    u32x4 *to = reinterpret_cast<u32x4 *>(out_val + head);
    for (uint32_t i = threadIdx.x; i < vecs; i += kMergeBlock) to[i] = zero;
    if (threadIdx.x < head) out_val[threadIdx.x] = O(0);
    for (uint32_t i = head + vecs * V + threadIdx.x; i < dense_n; i += kMergeBlock) out_val[i] = O(0);
  }
  uint32_t n = 0;
  if (slab_rank<kMergeBlock>(sh, geo, tie_bits, off, arr, live, rank, &n)) {
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i) {
      if (live & (1u << i)) {
        sh.key[rank[i]] = off[i];
        sh.tie[rank[i]] = __float_as_uint(KeyOf<S>::to_f32(v[i]));
      }
    }
  } else {
    (void)block_exclusive_scan<uint32_t, kMergeBlock>((uint32_t)__popc(live), sh.scan, &n);
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i)
      if (arr[i] < r) s_all.both[arr[i]] = live & (1u << i) ? ((uint64_t)off[i] << kMergeOneArrBits) | arr[i] : ~0ull;
    __syncthreads();
    sort_network(s_all.both, r);  // entries that are skipped come last
    uint64_t e[kMergeRecs];
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i) e[i] = arr[i] < n ? s_all.both[arr[i]] : 0ull;
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i) v[i] = val[(uint32_t)e[i] & ((1u << kMergeOneArrBits) - 1u)];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMergeRecs; ++i) {
      if (arr[i] < n) {
        sh.key[arr[i]] = (uint32_t)(e[i] >> kMergeOneArrBits);
        sh.tie[arr[i]] = __float_as_uint(KeyOf<S>::to_f32(v[i]));
      }
    }
  }
  __syncthreads();
  uint32_t k[kMergeItems];
  float sum[kMergeItems];
  // (a dense tensor takes every sum that is not zero, also one that rounds to -0)
  const uint32_t per = ((n + kMergeBlock - 1) / kMergeBlock) | 1u;  // as few places per thread as cover the list: <= kMergeItems
  const uint32_t keep = DENSE ? sum_runs<float>(sh, n, per, k, sum) : sum_runs<O>(sh, n, per, k, sum);
  uint32_t total;
  if (DENSE) wait_global_acks();  // this wave's zeros are written (the scan's barriers: everybody's)
  uint32_t at = block_exclusive_scan<uint32_t, kMergeBlock>((uint32_t)__popc(keep), sh.scan, &total);
#pragma unroll
  for (int q = 0; q < kMergeItems; ++q) {
    if (keep & (1u << q)) {
      if (DENSE) {
        out_val[k[q]] = SumAs<O>::of(sum[q]);
      } else {
        sh.key[at] = k[q];
        sh.tie[at] = __float_as_uint(sum[q]);
        ++at;
      }
    }
  }
  if (!DENSE) {
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < total; i += kMergeBlock) {
      if ((int64_t)i < capacity) {
        out_idx[i] = (I)sh.key[i];
        out_val[i] = SumAs<O>::of(__uint_as_float(sh.tie[i]));
      }
    }
    if (threadIdx.x == 0) {
      *out_count = (int64_t)total;
      if ((int64_t)total > capacity) atomicOr(status, ZEN_STAT_CAPACITY);
    }
  }
  if (answer.host) {
    wait_global_acks();  // its share of the status word, and the count
    __syncthreads();
    host_answer_count(answer, DENSE ? nullptr : out_count, status);
  }
}

// Entries up to which one workgroup does it all: as many as fit (6144 of them spread over the range 28 to 36 us a dense
// call, in the wide buckets' two launches 39).
constexpr int64_t kMergeOneMax = merge_one_max();
static_assert(kMergeOneMax <= kSlabCap, "the records fit");

template <typename S, typename O>
int merge_one_launch(const void *idx, int idx64_in, const S *val, int64_t r, int64_t dense_n, void *out_idx, int idx64_out,
                     O *out_val, int64_t capacity, int64_t *out_count, int32_t *status, hipStream_t s, const HostAsk &ask) {
  SlabGeom geo{};
  while ((dense_n >> geo.sub_shift) >= kSlabSubs) ++geo.sub_shift;  // 19 at most: with 13 bits of arrival number a word
  const int tie_bits = ceil_log2_u64((uint64_t)r);
  const dim3 grid(1), block(kMergeBlock);
  ProfScope prof(kProfWideMerge, s);
#define ZEN_ONE(I, DENSE)                                                                                             \
  k_merge_one<I, S, O, DENSE><<<grid, block, 0, s>>>(geo, idx, idx64_in, val, (uint32_t)r, (uint32_t)dense_n,         \
                                                     static_cast<I *>(out_idx), out_val, capacity, tie_bits, out_count, \
                                                     ask.answer, status)
  if (!out_idx)
    ZEN_ONE(int32_t, true);
  else if (idx64_out)
    ZEN_ONE(int64_t, false);
  else
    ZEN_ONE(int32_t, false);
#undef ZEN_ONE
  ZEN_LAUNCH_CHECK("k_merge_one");
  if (ask.answer.host) *ask.answered = true;
  return ZEN_OK;
}

// Memory that must be zero when a merge starts: the prefix state over the buckets and the scatter kernels'
// counters, for the largest geometry.  It sits at the head of the workspace whatever path a call takes, and a
// call on bucket slabs leaves it zero again, so that a caller who vouches for it (ZEN_MODE_ZEROED) saves the
// kernel that would clear it.
constexpr size_t kDoneBytes = (kDoneWords * sizeof(uint32_t) + 255) / 256 * 256;
constexpr size_t kMergeZeroBytes =
    ((scan_words_c(kSlabMaxBuckets) * sizeof(unsigned long long) + 255) / 256 * 256) +
    (size_t)kCoarseCursorWords * sizeof(uint32_t) + kDoneBytes + (size_t)kSlabMaxBuckets * sizeof(uint32_t);

struct SlabMergePlan {
  unsigned long long *scan;  // prefix state over the buckets (zeroed before use)
  uint32_t *done;            // [kDoneWords] buckets merged (the same)
  CoarseGeom cg;
  FeedBuffers feed;
  uint32_t *slab_idx, *slab_arr;
  void *slab_val;
  size_t zero_bytes;
  size_t bytes;
};

SlabMergePlan plan_slab_merge(void *workspace, const SlabGeom &geo, int64_t r) {  // sized for 4-byte values
  Carver cv(workspace);
  SlabMergePlan p;
  const size_t B = geo.nbuckets;
  p.scan = cv.take<unsigned long long>(scan_words((int64_t)B));
  p.feed.coarse_cursor = cv.take<uint32_t>(feed_coarse_cursor_words());
  p.done = cv.take<uint32_t>(kDoneWords);
  p.feed.cursor = cv.take<uint32_t>(B);
  p.zero_bytes = cv.used;
  cv.used = kMergeZeroBytes;  // whatever the geometry, the rest starts behind the largest zero region
  p.feed.bucket_lo = cv.take<uint32_t>(B);
  p.cg = coarse_geometry(geo, r);
  p.feed.coarse_words = cv.take<uint32_t>(feed_coarse_words(p.cg, 3));
  p.slab_idx = cv.take<uint32_t>(B * kSlabCap);
  p.slab_arr = cv.take<uint32_t>(B * kSlabCap);
  p.slab_val = cv.take<uint32_t>(B * kSlabCap);
  p.bytes = cv.used;
  return p;
}

bool slab_merge_fits(int64_t r, int64_t dense_n, SlabGeom *geo) {
  SlabGeom g;
  if (r < (1 << 15) || r > 0x7ffffffell || !slab_geometry(dense_n, 1, r, kMergeTarget, 0, &g)) return false;
  if (g.sub_shift + ceil_log2_u64((uint64_t)r) > 32) return false;  // (index inside a narrow range, arrival number) must fit a word
  if (geo) *geo = g;
  return true;
}

template <typename I, typename S, typename O>
int slab_merge_launch(const SlabGeom &geo, const I *idx, const S *val, int64_t r, int64_t dense_n, void *out_idx,
                      int idx64_out, O *out_val, int64_t capacity, int64_t *out_count, void *workspace,
                      bool zeroed, int32_t *status, hipStream_t s, const HostAsk &ask) {
  const SlabMergePlan p = plan_slab_merge(workspace, geo, r);
  if (!zeroed) {
    launch_fill<unsigned long long>(p.scan, 0ull, p.zero_bytes / sizeof(unsigned long long), s);
    ZEN_LAUNCH_CHECK("merge: clear prefix state");
  }
  {
    ProfScope prof(kProfMergeFeed, s);
    const MergeSrc<I, S> src{geo, idx, val, (uint32_t)dense_n, status};
    const MergeSink<S> sink{geo, p.slab_idx, p.slab_arr, static_cast<S *>(p.slab_val)};
    const int rc = feed_slabs<3>(geo, p.cg, src, sink, nullptr, r, p.feed, status, s);
    if (rc != ZEN_OK) return rc;
  }
  const ScanState st = scan_state(p.scan, (int64_t)geo.nbuckets);
  const int tie_bits = ceil_log2_u64((uint64_t)r);  // arrival numbers are < r
  ProfScope prof(kProfMergeBucket, s);
  if (idx64_out)
    k_merge_bucket<int64_t, S, O><<<dim3(geo.nbuckets), dim3(kMergeBlock), 0, s>>>(
        geo, p.feed.cursor, p.feed.coarse_cursor, p.feed.bucket_lo, p.slab_idx, p.slab_arr,
        static_cast<const S *>(p.slab_val), static_cast<int64_t *>(out_idx), out_val, capacity, st, p.done, tie_bits,
        out_count, ask.answer, status);
  else
    k_merge_bucket<int32_t, S, O><<<dim3(geo.nbuckets), dim3(kMergeBlock), 0, s>>>(
        geo, p.feed.cursor, p.feed.coarse_cursor, p.feed.bucket_lo, p.slab_idx, p.slab_arr,
        static_cast<const S *>(p.slab_val), static_cast<int32_t *>(out_idx), out_val, capacity, st, p.done, tie_bits,
        out_count, ask.answer, status);
  ZEN_LAUNCH_CHECK("k_merge_bucket");
  if (ask.answer.host) *ask.answered = true;
  return ZEN_OK;
}

struct MergePlan {
  uint32_t *keys, *tmp_v, *sort_k, *sort_v;
  void *scan;  // prefix state of the reduce kernel
  void *sort_scratch;
  size_t bytes;
  int ntiles;
};

MergePlan plan_merge(void *workspace, int64_t r, int64_t dense_n) {
  Carver cv(workspace);
  cv.used = kMergeZeroBytes;  // the head of the workspace belongs to the bucket-slab path's counters
  MergePlan p;
  const size_t cap = (size_t)(r > 0 ? r : 1);
  p.keys = cv.take<uint32_t>(cap);
  p.tmp_v = cv.take<uint32_t>(cap);
  p.sort_k = cv.take<uint32_t>(cap);
  p.sort_v = cv.take<uint32_t>(cap);
  p.ntiles = (int)ceil_div((int64_t)cap, kMrgTile);
  p.scan = cv.take<unsigned long long>(scan_words(p.ntiles));
  p.sort_scratch = cv.take<char>(sort_scratch_bytes((int64_t)cap));
  p.bytes = cv.used;
  SlabGeom geo;
  if (slab_merge_fits(r, dense_n, &geo)) {
    const size_t slabs = plan_slab_merge(nullptr, geo, r).bytes;
    if (slabs > p.bytes) p.bytes = slabs;
  }
  const size_t wide = wide_merge_bytes(r, dense_n, wide_device_cus());
  if (wide && kMergeZeroBytes + wide > p.bytes) p.bytes = kMergeZeroBytes + wide;
  return p;
}

// Whether a call with these sizes goes to one workgroup, to the wide buckets.
bool takes_one(int64_t r, int mode) { return (mode & 0xff) == ZEN_MODE_FAST && r <= kMergeOneMax; }
bool takes_wide(int64_t r, int64_t dense_n, int mode) {
  return (mode & ~ZEN_MODE_ZEROED) == ZEN_MODE_FAST && wide_merge_fits(r, dense_n, wide_device_cus(), nullptr);
}
// Whether the merge writes a dense tensor whole (one workgroup writes zeros at some 100 GB/s: up to 1 MB).
bool writes_dense(int64_t r, int64_t dense_n, int dtype, int mode) {
  return takes_one(r, mode) ? dense_n * (dtype == ZEN_BF16 ? 2 : 4) <= (1ll << 20) : takes_wide(r, dense_n, mode);
}

// O: float (the fp32 sums) or uint16_t (rounded once to bf16).  out_idx == nullptr: out_val is the dense tensor,
// written whole (where writes_dense says so).
template <typename S, typename O>
int merge_launch(const void *idx, int idx64_in, const S *val, int64_t r, int64_t dense_n, void *out_idx,
                 int idx64_out, O *out_val, int64_t capacity, int64_t *out_count, int mode, void *workspace,
                 int32_t *status, hipStream_t s, const HostAsk &ask = {}) {
  const bool zeroed = (mode & ZEN_MODE_ZEROED) != 0;
  if (takes_one(r, mode))
    return merge_one_launch(idx, idx64_in, val, r, dense_n, out_idx, idx64_out, out_val, capacity, out_count, status, s, ask);
  const bool wide = takes_wide(r, dense_n, mode);
  mode &= ~(ZEN_MODE_ZEROED | ZEN_MODE_SLABS);
  SlabGeom geo;
  if (wide) {
    // the zero region at the head of the workspace: the prefix state first, the cursors behind it
    Carver cv(workspace);
    unsigned long long *scan = cv.take<unsigned long long>(scan_words((int64_t)kSlabMaxBuckets));
    uint32_t *cursor = cv.take<uint32_t>(feed_coarse_cursor_words());
    uint32_t *done = cv.take<uint32_t>(kDoneWords);
    if (!zeroed) {
      launch_fill<unsigned long long>(scan, 0ull, kMergeZeroBytes / sizeof(unsigned long long), s);
      ZEN_LAUNCH_CHECK("merge: clear prefix state");
    }
    WideList list;
    if (!wide_merge_list(idx, idx64_in, val, r, dense_n, cursor, done, static_cast<char *>(workspace) + kMergeZeroBytes,
                         wide_device_cus(), status, &list, ask.answer.host != nullptr))
      return fail(ZEN_EINVAL, "zen_merge: sizes do not suit the wide buckets");
    return wide_merge(list, sizeof(S) == 2 ? ZEN_BF16 : ZEN_F32, out_idx, idx64_out, out_val,
                      sizeof(O) == 2 ? ZEN_BF16 : ZEN_F32, capacity, out_count, scan, s, ask);
  }
  if (mode == ZEN_MODE_FAST && slab_merge_fits(r, dense_n, &geo)) {
    if (idx64_in)
      return slab_merge_launch(geo, static_cast<const int64_t *>(idx), val, r, dense_n, out_idx, idx64_out, out_val,
                               capacity, out_count, workspace, zeroed, status, s, ask);
    return slab_merge_launch(geo, static_cast<const int32_t *>(idx), val, r, dense_n, out_idx, idx64_out, out_val,
                             capacity, out_count, workspace, zeroed, status, s, ask);
  }
  MergePlan p = plan_merge(workspace, r, dense_n);
  const unsigned blocks = (unsigned)ceil_div(r, 256);
  launch_fill<unsigned long long>(static_cast<unsigned long long *>(p.scan), 0ull, scan_words(p.ntiles), s);
  {
    ProfScope prof(kProfMergePrep, s);
    if (idx64_in)
      k_merge_prep<int64_t, S><<<dim3(blocks), dim3(256), 0, s>>>(static_cast<const int64_t *>(idx), val, (uint32_t)r,
                                                                  (uint32_t)dense_n, p.keys, p.tmp_v, status);
    else
      k_merge_prep<int32_t, S><<<dim3(blocks), dim3(256), 0, s>>>(static_cast<const int32_t *>(idx), val, (uint32_t)r,
                                                                  (uint32_t)dense_n, p.keys, p.tmp_v, status);
    ZEN_LAUNCH_CHECK("k_merge_prep");
  }
  const uint32_t *sk, *sp;
  {
    // fast mode: indices that a hash assigned to one destination spread evenly over the dense length, so
    // the bucket sort applies; a crowded key range makes it raise ZEN_STAT_RETRY
    ProfScope prof(kProfSort, s);
    int where;
    if (mode == ZEN_MODE_FAST && bucket_sort_fits(r, (uint32_t)dense_n))
      where = bucket_sort_pairs(p.keys, p.tmp_v, p.sort_k, p.sort_v, r, nullptr, (uint32_t)dense_n, p.sort_scratch,
                                status, s);
    else
      where = sort_pairs(p.keys, p.tmp_v, p.sort_k, p.sort_v, r, nullptr, ceil_log2_u64((uint64_t)dense_n),
                         p.sort_scratch, status, s);
    if (where < 0) return where;
    sk = where ? p.sort_k : p.keys;
    sp = where ? p.sort_v : p.tmp_v;
  }
  const ScanState st = scan_state(p.scan, p.ntiles);
  ProfScope prof(kProfMergeReduce, s);
  if (idx64_out)
    k_merge_reduce<int64_t, O><<<dim3((unsigned)p.ntiles), dim3(kMrgBlock), 0, s>>>(
        sk, sp, (uint32_t)r, (uint32_t)dense_n, static_cast<int64_t *>(out_idx), out_val, capacity, st, p.ntiles,
        out_count, status);
  else
    k_merge_reduce<int32_t, O><<<dim3((unsigned)p.ntiles), dim3(kMrgBlock), 0, s>>>(
        sk, sp, (uint32_t)r, (uint32_t)dense_n, static_cast<int32_t *>(out_idx), out_val, capacity, st, p.ntiles,
        out_count, status);
  ZEN_LAUNCH_CHECK("k_merge_reduce");
  return ZEN_OK;
}

int merge_check(const void *idx, const void *val, int dtype, int64_t r, int64_t dense_n, int mode, const char **why) {
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) { *why = "bad dtype"; return ZEN_EINVAL; }
  if ((mode & ~(ZEN_MODE_ZEROED | ZEN_MODE_SLABS)) != ZEN_MODE_FAST &&
      (mode & ~(ZEN_MODE_ZEROED | ZEN_MODE_SLABS)) != ZEN_MODE_GENERAL) {
    *why = "bad mode";
    return ZEN_EINVAL;
  }
  if (r < 0 || r > 0x7ffffffell || dense_n <= 0 || dense_n > 0x7fffffffll) {
    *why = "need 0 <= r < 2^31 - 1 and 0 < dense_n < 2^31";
    return ZEN_EINVAL;
  }
  if (r > 0 && (!idx || !val)) { *why = "null pointer"; return ZEN_EINVAL; }
  return ZEN_OK;
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_merge_workspace(int64_t r, int64_t dense_n) {
  if (r < 0 || dense_n <= 0) return 0;
  return zen::plan_merge(nullptr, r, dense_n).bytes;
}

size_t zen_merge_zero_bytes(void) { return zen::kMergeZeroBytes; }

int zen_merge_path(int64_t r, int64_t dense_n, int mode) {
  const bool slabs_only = (mode & ZEN_MODE_SLABS) != 0;
  mode &= ~(ZEN_MODE_ZEROED | ZEN_MODE_SLABS);
  if (mode != ZEN_MODE_FAST || r <= 0 || dense_n <= 0) return 0;
  if (!slabs_only && zen::wide_merge_fits(r, dense_n, zen::wide_device_cus(), nullptr)) return 3;
  if (zen::slab_merge_fits(r, dense_n, nullptr)) return 2;
  return zen::bucket_sort_fits(r, (uint32_t)dense_n) ? 1 : 0;
}

}  // extern "C"

namespace {

int merge_call(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, int64_t dense_n, void *out_idx,
               int idx64_out, void *out_val, bool round, int64_t capacity, int64_t *out_count, int mode,
               void *workspace, size_t workspace_bytes, int32_t *status, void *stream, const zen::HostAsk &ask = {}) {
  using namespace zen;
  const char *why = "";
  if (merge_check(idx, val, dtype, r, dense_n, mode, &why) != ZEN_OK) return fail(ZEN_EINVAL, why);
  if (!out_count || !status || capacity < 0) return fail(ZEN_EINVAL, "zen_merge: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (r == 0) {
    launch_fill<int64_t>(out_count, 0, 1, s);
    ZEN_LAUNCH_CHECK("zen_merge: zero count");
    return ZEN_OK;
  }
  if (!workspace || (capacity > 0 && (!out_idx || !out_val))) return fail(ZEN_EINVAL, "zen_merge: null pointer");
  if (workspace_bytes < zen_merge_workspace(r, dense_n)) return fail(ZEN_EWORKSPACE, "zen_merge: workspace too small");
  if (dtype == ZEN_BF16 && round)
    return merge_launch(idx, idx64_in, static_cast<const uint16_t *>(val), r, dense_n, out_idx, idx64_out,
                        static_cast<uint16_t *>(out_val), capacity, out_count, mode, workspace, status, s, ask);
  if (dtype == ZEN_BF16)
    return merge_launch(idx, idx64_in, static_cast<const uint16_t *>(val), r, dense_n, out_idx, idx64_out,
                        static_cast<float *>(out_val), capacity, out_count, mode, workspace, status, s, ask);
  return merge_launch(idx, idx64_in, static_cast<const uint32_t *>(val), r, dense_n, out_idx, idx64_out,
                      static_cast<float *>(out_val), capacity, out_count, mode, workspace, status, s, ask);
}

}  // namespace

extern "C" {

int zen_merge(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, int64_t dense_n, void *out_idx,
              int idx64_out, float *out_val, int64_t capacity, int64_t *out_count, int mode, void *workspace,
              size_t workspace_bytes, int32_t *status, void *stream) {
  return merge_call(idx, idx64_in, val, dtype, r, dense_n, out_idx, idx64_out, out_val, false, capacity, out_count,
                    mode, workspace, workspace_bytes, status, stream);
}

int zen_merge_rounded(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, int64_t dense_n,
                      void *out_idx, int idx64_out, void *out_val, int64_t capacity, int64_t *out_count, int mode,
                      void *workspace, size_t workspace_bytes, int32_t *status, void *stream) {
  return merge_call(idx, idx64_in, val, dtype, r, dense_n, out_idx, idx64_out, out_val, true, capacity, out_count,
                    mode, workspace, workspace_bytes, status, stream);
}

int zen_merge_rounded_count(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, int64_t dense_n,
                            void *out_idx, int idx64_out, void *out_val, int64_t capacity, int64_t *out_count, int mode,
                            void *workspace, size_t workspace_bytes, int32_t *status, int64_t *host, int64_t words,
                            void *stream) {
  using namespace zen;
  HostAnswer answer;
  bool answered = false;
  int rc = host_ask(host, words, 2, &answer);
  if (rc != ZEN_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = merge_call(idx, idx64_in, val, dtype, r, dense_n, out_idx, idx64_out, out_val, true, capacity, out_count, mode,
                  workspace, workspace_bytes, status, stream, HostAsk{answer, &answered});
  if (rc == ZEN_OK && !answered) rc = host_answer_launch(answer, out_count, 1, status, 1, s);
  return host_finish(rc, answer, s);
}

size_t zen_decode_dense_workspace(int64_t r, int64_t dense_n) {
  if (r < 0 || dense_n <= 0) return 0;
  const size_t cap = (size_t)(r > 0 ? r : 1);
  return zen::align_up(cap * sizeof(int32_t), 256) + zen::align_up(cap * sizeof(float), 256) + 256 +
         zen::align_up(zen_merge_workspace(r, dense_n), 256);
}

}  // extern "C"

namespace zen {
namespace {

int decode_call(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, void *dense, int64_t dense_n,
                int mode, void *workspace, size_t workspace_bytes, int32_t *status, void *stream,
                const HostAsk &ask = {}) {
  const char *why = "";
  if (merge_check(idx, val, dtype, r, dense_n, mode, &why) != ZEN_OK) return fail(ZEN_EINVAL, why);
  if (!dense || !status) return fail(ZEN_EINVAL, "zen_decode_dense: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // the zero region zen_merge wants is at the head of this call's workspace too
  Carver cv(workspace);
  void *inner = cv.take<char>(zen_merge_workspace(r, dense_n));
  const bool whole = r > 0 && writes_dense(r, dense_n, dtype, mode);  // the merge writes the dense tensor, zeros included
  if (r > 0 && !workspace) return fail(ZEN_EINVAL, "zen_decode_dense: null pointer");
  if (r > 0 && workspace_bytes < zen_decode_dense_workspace(r, dense_n))
    return fail(ZEN_EWORKSPACE, "zen_decode_dense: workspace too small");
  if (whole) {
    if (dtype == ZEN_BF16)
      return merge_launch(idx, idx64_in, static_cast<const uint16_t *>(val), r, dense_n, nullptr, 0,
                          static_cast<uint16_t *>(dense), r, nullptr, mode, inner, status, s, ask);
    return merge_launch(idx, idx64_in, static_cast<const uint32_t *>(val), r, dense_n, nullptr, 0,
                        static_cast<float *>(dense), r, nullptr, mode, inner, status, s, ask);
  }
  if (dtype == ZEN_BF16)
    launch_fill<uint16_t>(static_cast<uint16_t *>(dense), (uint16_t)0, (size_t)dense_n, s);
  else
    launch_fill<uint32_t>(static_cast<uint32_t *>(dense), 0u, (size_t)dense_n, s);
  ZEN_LAUNCH_CHECK("zen_decode_dense: clear");
  if (r == 0) return ZEN_OK;
  int32_t *m_idx = cv.take<int32_t>((size_t)r);
  float *m_val = cv.take<float>((size_t)r);
  int64_t *m_count = cv.take<int64_t>(1);
  int rc;
  if (dtype == ZEN_BF16)
    rc = merge_launch(idx, idx64_in, static_cast<const uint16_t *>(val), r, dense_n, m_idx, 0, m_val, r, m_count, mode,
                      inner, status, s);
  else
    rc = merge_launch(idx, idx64_in, static_cast<const uint32_t *>(val), r, dense_n, m_idx, 0, m_val, r, m_count, mode,
                      inner, status, s);
  if (rc != ZEN_OK) return rc;
  const unsigned blocks = (unsigned)ceil_div(r, 256);
  if (dtype == ZEN_BF16)
    k_scatter_dense<uint16_t><<<dim3(blocks), dim3(256), 0, s>>>(m_idx, m_val, m_count, static_cast<uint16_t *>(dense),
                                                                 (uint32_t)dense_n);
  else
    k_scatter_dense<uint32_t><<<dim3(blocks), dim3(256), 0, s>>>(m_idx, m_val, m_count, static_cast<uint32_t *>(dense),
                                                                 (uint32_t)dense_n);
  ZEN_LAUNCH_CHECK("k_scatter_dense");
  return ZEN_OK;
}

}  // namespace
}  // namespace zen

extern "C" {

int zen_decode_dense(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, void *dense,
                     int64_t dense_n, int mode, void *workspace, size_t workspace_bytes, int32_t *status,
                     void *stream) {
  return zen::decode_call(idx, idx64_in, val, dtype, r, dense, dense_n, mode, workspace, workspace_bytes, status, stream);
}

int zen_decode_dense_status(const void *idx, int idx64_in, const void *val, int dtype, int64_t r, void *dense,
                            int64_t dense_n, int mode, void *workspace, size_t workspace_bytes, int32_t *status,
                            int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  bool answered = false;
  int rc = host_ask(host, words, 1, &answer);
  if (rc != ZEN_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = decode_call(idx, idx64_in, val, dtype, r, dense, dense_n, mode, workspace, workspace_bytes, status, stream,
                   HostAsk{answer, &answered});
  if (rc == ZEN_OK && !answered) rc = host_answer_launch(answer, nullptr, 0, status, 1, s);
  return host_finish(rc, answer, s);
}

}  // extern "C"

namespace zen {
namespace {

// The merged entries on their way to the second exchange (comm.py:125-127 turns the dense fp32 sums into the
// tensor's type and takes the nonzeros again): every sum is rounded once to the type V, entries whose sum
// rounds to zero are dropped, the others keep their order.  One pass: a tile of kRcBlock * kRcItems entries per
// workgroup, the tiles' kept counts chained by look-back.  count sits on the device.
constexpr int kRcBlock = 256, kRcItems = 8, kRcTile = kRcBlock * kRcItems;
template <typename I, typename V>
__global__ __launch_bounds__(kRcBlock) void k_round_compact(const I *__restrict__ idx, const float *__restrict__ sums,
                                                            const int64_t *__restrict__ count, int64_t capacity,
                                                            I *__restrict__ out_idx, V *__restrict__ out_val,
                                                            int64_t *out_count, ScanState st, int32_t *status) {
  __shared__ uint32_t tile_s;
  __shared__ uint32_t scan_s[kRcBlock / 64 + 1];
  __shared__ uint64_t base_s;
  if (threadIdx.x == 0) tile_s = atomicAdd(st.ticket, 1u);
  __syncthreads();
  const uint32_t tile = tile_s;
  int64_t n = *count;
  if (n > capacity) n = capacity;
  const int64_t first = (int64_t)tile * kRcTile + (int64_t)threadIdx.x * kRcItems;
  I k[kRcItems];
  V v[kRcItems];
  uint32_t keep = 0, mine = 0;
#pragma unroll
  for (int i = 0; i < kRcItems; ++i) {
    const int64_t j = first + i;
    k[i] = 0;
    v[i] = 0;
    if (j < n) {
      k[i] = idx[j];
      const float f = sums[j];
      if constexpr (sizeof(V) == 2) {
        v[i] = f32_to_bf16_rne(f);
        if (v[i] & 0x7fffu) keep |= 1u << i;
      } else {
        v[i] = __float_as_uint(f);
        if (v[i] & 0x7fffffffu) keep |= 1u << i;
      }
    }
  }
  mine = __popc(keep);
  uint32_t total;
  const uint32_t before = block_exclusive_scan<uint32_t, kRcBlock>(mine, scan_s, &total);
  const uint64_t base = lookback_exclusive(st, (int)tile, total, status, &base_s);
  uint64_t at = base + before;
#pragma unroll
  for (int i = 0; i < kRcItems; ++i)
    if (keep & (1u << i)) {
      out_idx[at] = k[i];
      out_val[at] = v[i];
      ++at;
    }
  if (tile == gridDim.x - 1 && threadIdx.x == kRcBlock - 1) *out_count = (int64_t)(base + before + mine);
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_round_compact_workspace(int64_t capacity) {
  if (capacity < 0) return 0;
  return zen::scan_words(zen::ceil_div(capacity > 0 ? capacity : 1, (int64_t)zen::kRcTile)) * sizeof(uint64_t);
}

int zen_round_compact(const void *idx, int idx64, const float *sums, const int64_t *count, int64_t capacity, int dtype,
                      void *out_idx, void *out_val, int64_t *out_count, void *workspace, size_t workspace_bytes,
                      int32_t *status, void *stream) {
  using namespace zen;
  if (!count || !out_count || !status || capacity < 0) return fail(ZEN_EINVAL, "zen_round_compact: null pointer");
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_round_compact: bad dtype");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (capacity == 0) {
    launch_fill<int64_t>(out_count, 0, 1, s);
    ZEN_LAUNCH_CHECK("zen_round_compact: zero count");
    return ZEN_OK;
  }
  if (!idx || !sums || !out_idx || !out_val || !workspace) return fail(ZEN_EINVAL, "zen_round_compact: null pointer");
  if (workspace_bytes < zen_round_compact_workspace(capacity))
    return fail(ZEN_EWORKSPACE, "zen_round_compact: workspace too small");
  const int64_t tiles = ceil_div(capacity, (int64_t)kRcTile);
  if (tiles > 0x7fffffffll) return fail(ZEN_EINVAL, "zen_round_compact: too many entries");
  launch_fill<uint64_t>(static_cast<uint64_t *>(workspace), 0ull, scan_words(tiles), s);
  ZEN_LAUNCH_CHECK("zen_round_compact: clear");
  const ScanState st = scan_state(workspace, tiles);
  const dim3 grid((unsigned)tiles), block(kRcBlock);
#define ZEN_RC(I, V)                                                                                              \
  k_round_compact<I, V><<<grid, block, 0, s>>>(static_cast<const I *>(idx), sums, count, capacity,              \
                                               static_cast<I *>(out_idx), static_cast<V *>(out_val), out_count, \
                                               st, status)
  if (idx64) {
    if (dtype == ZEN_BF16) ZEN_RC(int64_t, uint16_t); else ZEN_RC(int64_t, uint32_t);
  } else {
    if (dtype == ZEN_BF16) ZEN_RC(int32_t, uint16_t); else ZEN_RC(int32_t, uint32_t);
  }
#undef ZEN_RC
  ZEN_LAUNCH_CHECK("k_round_compact");
  return ZEN_OK;
}

}  // extern "C"
