// Receive side on wide buckets (zen_wide.h): the fast path of zen_merge for a few million received entries at
// most.
//
// The reference builds a dense zero tensor of the full gradient length, scatter-adds every payload into it
// and extracts the nonzeros again (comm.py:32-50).  The indices a destination receives were assigned to it by
// a hash, so they spread evenly over [0, dense_n): the entries go to at most 256 buckets by index range, as
// (index, arrival number, value) records (k_wide_scatter: a workgroup orders its 4096 entries by bucket in
// LDS and writes one run per bucket), and one workgroup per bucket sorts its bucket by (index, arrival number)
// inside LDS, sums every run of equal indices in arrival order from +0 (bit-identical to a sequential
// scatter_add_), drops zero sums and writes what is left at the place the buckets before it leave off
// (k_wide_merge).  Two launches; zen_merge.hip needs three, and a thousand buckets, for the same input.
#include "zen_wide.h"

namespace zen {
namespace {

constexpr int kWmRounds = 3;                               // a part of a bucket's slab is read in rounds of kWideBlock records
constexpr int kWmPartMax = kWideBlock * kWmRounds;         // records of one part, at most
constexpr int kWmLanes = 4;                                // records a thread handles per step of the ranking loops
constexpr int kWmQueue = 6144;                             // records of large groups set aside while ranking
constexpr int kWmGroupLimit = 2048;                        // records in one narrow range: bounds the rank loop
constexpr int kWmSumItems = 17;                            // sorted records per thread while summing, at most (odd: no LDS bank conflicts)
constexpr int kWmPad = 20;                                 // words behind the records that may be read, not looked at
constexpr uint32_t kInvalid = 0xffffffffu;
static_assert(kWideBlock * kWmSumItems >= kWideCap, "every sorted place needs an owner");
static_assert(kWmQueue <= (1 << 14) && kWideCap <= (1 << 14) && kWideSubs <= (1 << 14), "queue entries in one word");

// ------------------------------------------------------------ list -> buckets

constexpr int kWsBlock = 512;
constexpr int kWsItems = 8;
constexpr int kWsBatch = kWsBlock * kWsItems;  // list entries per workgroup

template <typename S>
__global__ __launch_bounds__(kWsBlock) void k_wide_scatter(WideList list) {
  // 32 KB of LDS: five workgroups share a compute unit and the whole grid is resident in one round (the values
  // do not pass through LDS for that reason: they are fetched again when the record is written)
  __shared__ WideScatterShared<kWsBlock, kWsItems> sh;
  wide_scatter_prepare(list, sh);
  wide_scatter_batch<S>(list, blockIdx.x, blockIdx.x % kWideSplit, sh);
}

// ------------------------------------------------------------ a bucket

struct WideMergeShared {
  union {
    uint32_t word[kWideCap + kWmPad];  // while ranking: (index inside its narrow range) << tie_bits | arrival number
    uint32_t key[kWideCap + kWmPad];   // afterwards: the sorted indices (minus the bucket's first), then the kept ones
  };
  union {
    WideCounters cnt;
    float val[kWideCap + kWmPad];      // the sorted values, then the kept sums
  };
  uint32_t queue[kWmQueue];   // records set aside: place in `word` | narrow range << 14, then the rank
  uint32_t scan[kWideBlock / 64 + 1];
  uint32_t qn, big;
  int tile;
};

// Puts the bucket's records in order of (index, arrival number): indices (minus the bucket's first) to sh.key, values to
// sh.val.  Returns how many there are.  ROUNDS: of kWideBlock records of every part.  Up to two are written out, a thread's
// (at most sixteen) records stay in registers from their load to the end, and all loads are in flight together; of three
// the loops' bodies handle the first kWmLanes registers of a set and then rotate the set, and the values are loaded at the
// end (written out for 24 records the code would not fit the instruction cache, and every workgroup runs it once).  A
// chain of trips to LDS and memory: 62 M bf16, 3.1 M entries, 256 buckets of two rounds 39.2 us to index lists and 52.1
// dense at the time (42.6 and 55.0 before, with the loops for those too 48.2 and 59.0); 9 M, 0.9 M entries, one round 26.8 and 32.4.
template <typename S, int ROUNDS, typename Zero>
__device__ inline uint32_t wide_merge_sort(WideMergeShared &sh, const SlabGeom &geo, const WideSlabs &in, uint32_t b,
                                           const uint32_t (&pcount)[kWideSplit], uint32_t longest, bool declined,
                                           int tie_bits, int32_t *status, Zero zero_some) {
  constexpr int kItems = kWideSplit * ROUNDS, kSteps = kItems / kWmLanes;
  constexpr bool kHeld = ROUNDS <= 2;
  const uint32_t tid = threadIdx.x;
  const uint2 *rec_plane = in.rec + (size_t)b * kWideSplit * in.part_cap;
  const uint32_t *val_plane = in.val32 + (size_t)b * kWideSplit * in.part_cap;
  const int shift = geo.sub_shift;
  const uint32_t low_mask = (1u << shift) - 1u;

  // item r * kWideSplit + q of a thread is the record at place wide_place(q) + r * kWideBlock of part q; loads in no
  // branch, so that all are in flight together
  uint32_t w[kItems], ps[kItems];  // the record's word; then its place in `word` | narrow range << 14
  uint32_t v[kHeld ? kItems : 1];
  if (kHeld) {
    uint2 rec[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const uint32_t e = wide_place(i % kWideSplit) + (uint32_t)(i / kWideSplit) * kWideBlock;
      const size_t at = (size_t)(i % kWideSplit) * in.part_cap + (e < pcount[i % kWideSplit] ? e : 0u);
      rec[i] = rec_plane[at];
      v[kHeld ? i : 0] = sizeof(S) == 2 ? 0u : val_plane[at];
    }
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const bool live = wide_place(i % kWideSplit) + (uint32_t)(i / kWideSplit) * kWideBlock < pcount[i % kWideSplit];
      const uint32_t off = wm_off(rec[i]), arr = wm_arr(rec[i]);
      w[i] = live ? ((off & low_mask) << tie_bits) | arr : kInvalid;
      ps[i] = live ? off >> shift : kInvalid;  // the narrow range, for now
      if (sizeof(S) == 2) v[kHeld ? i : 0] = rec[i].y >> 16;
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
#pragma unroll
      for (int q = 0; q < kWideSplit; ++q) w[r * kWideSplit + q] = ps[r * kWideSplit + q] = kInvalid;
      if ((uint32_t)r * kWideBlock < longest) {
#pragma unroll
        for (int q = 0; q < kWideSplit; ++q) {
          const uint32_t e = wide_place(q) + (uint32_t)r * kWideBlock;
          const bool live = e < pcount[q];
          const uint2 rec = rec_plane[(size_t)q * in.part_cap + (live ? e : 0u)];
          const uint32_t off = wm_off(rec), arr = wm_arr(rec);
          if (live) {
            w[r * kWideSplit + q] = ((off & low_mask) << tie_bits) | arr;
            ps[r * kWideSplit + q] = off >> shift;
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i)
    if (ps[i] != kInvalid) sh.cnt.count(ps[i]);
  __syncthreads();
  uint32_t n = sh.cnt.starts(sh.scan, (uint32_t)kWmGroupLimit, &sh.big);
  __syncthreads();
  if (n > (uint32_t)kWideCap || sh.big) {  // more than fits, or keys piled on a few values: another path answers
    declined = true;
    __syncthreads();
    sh.cnt.clear();
#pragma unroll
    for (int i = 0; i < kItems; ++i) w[i] = ps[i] = kInvalid;
    n = 0;
    longest = 0;
    __syncthreads();
  }
  if (declined && tid == 0) atomicOr(status, ZEN_STAT_RETRY);
  // this workgroup was the only reader of its part cursors: back to zero for the next call
  if (tid < (uint32_t)kWideSplit) in.cursor[coarse_cursor_at(b, tid)] = 0;

  auto rotate = [](uint32_t (&a)[kItems]) {
    uint32_t head[kWmLanes];
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) head[k] = a[k];
#pragma unroll
    for (int i = 0; i + kWmLanes < kItems; ++i) a[i] = a[i + kWmLanes];
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) a[kItems - kWmLanes + k] = head[k];
  };
  const int steps = longest == 0 ? 0 : (int)((longest + kWideBlock - 1) / kWideBlock) * (kWideSplit / kWmLanes);
  auto take_step = [&](int from) {
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) {
      if (ps[from + k] != kInvalid) {
        const uint32_t p = sh.cnt.take(ps[from + k]);
        sh.word[p] = w[from + k];
        ps[from + k] = p | (ps[from + k] << 14);
      }
    }
  };
  if (kHeld) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (s < steps) take_step(s * kWmLanes);
      zero_some();
    }
  } else {
#pragma unroll 1
    for (int s = 0; s < kSteps; ++s) {
      if (s < steps) take_step(0);
      rotate(w);
      rotate(ps);
      zero_some();
    }
  }
  __syncthreads();
  // rank = records of the bucket with a smaller (index, arrival number): those of the narrow ranges before,
  // plus those of the record's own range with a smaller word.  The range's first four words are fetched in one
  // go, which settles ranges up to that size; where many records share an index (payloads that overlap) a few
  // lanes of every wave would walk through dozens of words while the others wait: records of larger ranges
  // are set aside and handed out again afterwards, one per thread.
  uint32_t rk[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i) rk[i] = kInvalid;
  auto rank_step = [&](int from, uint32_t (&out)[kWmLanes]) {
    constexpr int kAhead = 4;
    bool some = false;
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) some |= ps[from + k] != kInvalid;
    if (!__any(some)) return;
    uint32_t g0[kWmLanes], g1[kWmLanes], a[kWmLanes][kAhead];
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) {
      const uint32_t sub = ps[from + k] != kInvalid ? ps[from + k] >> 14 : 0u;
      g0[k] = sh.cnt.start_of(sub);
      g1[k] = sh.cnt.end_of(sub);
    }
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) {
#pragma unroll
      for (int e = 0; e < kAhead; ++e) a[k][e] = sh.word[g0[k] + e];  // what lies behind the range is not looked at
    }
#pragma unroll
    for (int k = 0; k < kWmLanes; ++k) {
      if (ps[from + k] != kInvalid) {
        const uint32_t size = g1[k] - g0[k];
        uint32_t less = a[k][0] < w[from + k] ? 1u : 0u;
#pragma unroll
        for (int e = 1; e < kAhead; ++e) less += ((size > (uint32_t)e) & (a[k][e] < w[from + k])) ? 1u : 0u;
        uint32_t x = g0[k] + less;
        if (size > (uint32_t)kAhead) {
          const uint32_t at = atomicAdd(&sh.qn, 1u);
          if (at < (uint32_t)kWmQueue) {
            sh.queue[at] = ps[from + k];
            x = 0x80000000u | at;  // pending: place in the queue
          } else {  // no room to set it aside: walked through here
            for (uint32_t u = g0[k] + kAhead; u < g1[k]; ++u) x += sh.word[u] < w[from + k];
          }
        }
        out[k] = x;
      }
    }
  };
  if (kHeld) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      uint32_t out[kWmLanes];
#pragma unroll
      for (int k = 0; k < kWmLanes; ++k) out[k] = kInvalid;
      if (s < steps) rank_step(s * kWmLanes, out);
#pragma unroll
      for (int k = 0; k < kWmLanes; ++k) rk[s * kWmLanes + k] = out[k];
      zero_some();
    }
  } else {
#pragma unroll 1
    for (int s = 0; s < kSteps; ++s) {
      uint32_t out[kWmLanes];
#pragma unroll
      for (int k = 0; k < kWmLanes; ++k) out[k] = kInvalid;
      if (s < steps) rank_step(0, out);
      rotate(w);
      rotate(ps);
      rotate(rk);  // the step's ranks enter at the end: after the last step rank i belongs to record i
#pragma unroll
      for (int k = 0; k < kWmLanes; ++k) rk[kItems - kWmLanes + k] = out[k];
      zero_some();
    }
  }
  __syncthreads();
  {
    uint32_t pending = sh.qn;
    if (pending > (uint32_t)kWmQueue) pending = kWmQueue;
    for (uint32_t e = tid; e < pending; e += kWideBlock) {
      const uint32_t p = sh.queue[e] & 0x3fffu, sub = sh.queue[e] >> 14;
      const uint32_t g0 = sh.cnt.start_of(sub), g1 = sh.cnt.end_of(sub);
      const uint32_t less = count_less(sh.word, g0, g1, sh.word[p]);
      sh.queue[e] = g0 + less;  // the entry's thread is its only reader
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; ++i)
      if (rk[i] != kInvalid && (rk[i] & 0x80000000u)) rk[i] = sh.queue[rk[i] & 0x7fffffffu];
  }
  __syncthreads();  // everybody is through with the words and the counters: the sorted records take their place
  if (kHeld) {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      if (rk[i] != kInvalid) {
        sh.key[rk[i]] = ((ps[i] >> 14) << shift) | (w[i] >> tie_bits);
        sh.val[rk[i]] = KeyOf<S>::to_f32((S)v[kHeld ? i : 0]);
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      if ((uint32_t)r * kWideBlock < longest) {
        uint32_t u[kWideSplit];
#pragma unroll
        for (int q = 0; q < kWideSplit; ++q) {
          const bool live = rk[r * kWideSplit + q] != kInvalid;
          const uint32_t e = wide_place(q) + (uint32_t)r * kWideBlock;
          const size_t at = (size_t)q * in.part_cap + (live ? e : 0u);
          u[q] = sizeof(S) == 2 ? rec_plane[at].y >> 16 : val_plane[at];
        }
#pragma unroll
        for (int q = 0; q < kWideSplit; ++q) {
          const int i = r * kWideSplit + q;
          if (rk[i] != kInvalid) {
            sh.key[rk[i]] = ((ps[i] >> 14) << shift) | (w[i] >> tie_bits);
            sh.val[rk[i]] = KeyOf<S>::to_f32((S)u[q]);
          }
        }
      }
    }
  }
  __syncthreads();
  return n;
}

// The sums of the n sorted records, what is kept of them put side by side to sh.key (plus `lo`) / sh.val (visible behind a
// barrier); returns how many.  publish(total) is called before they are put there.  Thread t owns the sorted places
// [t * ITEMS, (t + 1) * ITEMS), fetches them all at once (also what lies behind the last one, which counts for nothing) and
// walks through them in registers.  A run of equal indices is summed in arrival order from +0 (like the dense
// tensor of comm.py:35) and belongs to the thread that holds its last record; where that run began before
// the thread's first place (rare: runs are short next to ITEMS, long ones come from payloads that overlap),
// the part in front is summed first, from the run's head on.  Bound by vector instructions with four waves to a SIMD to
// hide them: 218 for every record and lane with places for a full bucket in every one, checks on every word read ahead and
// ranges that took five instructions to find; 62 M bf16, 3.1 M entries, 256 buckets of 12 000 records 38.0 -> 34.7 us, dense
// 51.5 -> 48.8; 268 M, 2.7 M entries 36.6 -> 33.0; 0.3 M entries in 128 buckets beside the encode 17.4 -> 14.5.
template <typename O, bool DENSE, int ITEMS, typename Publish>
__device__ __forceinline__ uint32_t wide_merge_sums(WideMergeShared &sh, uint32_t n, uint32_t lo, Publish publish) {
  static_assert(ITEMS <= kWmPad && ITEMS % 2 == 1, "words behind the records");
  constexpr uint32_t kNoKey = 0xffffffffu;  // offsets are below the bucket width
  const uint32_t first = threadIdx.x * (uint32_t)ITEMS;
  const uint32_t left = first < n ? n - first : 0u;
  const uint32_t own = left < (uint32_t)ITEMS ? left : (uint32_t)ITEMS;
  const uint32_t from = first < (uint32_t)kWideCap ? first : (uint32_t)kWideCap;
  uint32_t k[ITEMS];
  float sum[ITEMS];
  uint32_t keep = 0;
  {
    float v[ITEMS];
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
      k[q] = sh.key[from + q];
      v[q] = sh.val[from + q];
    }
    const uint32_t before = sh.key[from > 0 ? from - 1u : 0u], after = sh.key[first + ITEMS < n ? first + ITEMS : 0u];
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) k[q] = (uint32_t)q < own ? k[q] : kNoKey;
    const uint32_t before_k = first > 0 ? before : kNoKey;
    const uint32_t after_k = first + ITEMS < n ? after : kNoKey;
    float acc = 0.0f;
    if (own && before_k == k[0]) {
      // the run began before this thread's places: find its head, sum up to the place in front of `first`
      acc = sum_run_before(sh.key, sh.val, first, before_k);
    }
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
      const uint32_t prev = q > 0 ? k[q > 0 ? q - 1 : 0] : before_k;
      const uint32_t next = q + 1 < ITEMS ? k[q + 1 < ITEMS ? q + 1 : q] : after_k;
      acc = (k[q] != prev ? 0.0f : acc) + v[q];
      sum[q] = acc;
      keep |= (((uint32_t)q < own) & (k[q] != next) & (DENSE ? acc != 0.0f : SumAs<O>::kept(acc))) ? 1u << q : 0u;
    }
  }
  if (DENSE) wait_global_acks();  // this wave's zeros are written (the scan's barrier: everybody's)
  uint32_t total;
  uint32_t li = block_exclusive_scan<uint32_t, kWideBlock>((uint32_t)__popc(keep), sh.scan, &total);
  publish(total);
  // everybody is past reading the sorted bucket: the scan synchronised
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    if (keep & (1u << q)) {
      sh.key[li] = k[q] + lo;
      sh.val[li] = sum[q];
      ++li;
    }
  }
  return total;
}

// O: what is written for a sum (zen_common.h).  DENSE: out_val is the dense tensor [0, dense_n); the workgroup
// writes its bucket's range of it whole, zeros between the steps of the ranking loops, the sums behind them at the
// end (62 M bf16 elements, 3.1 M entries: 55 us; nine more with the zeros in front of the records' loads, which then wait for
// them to be written; the fill and scatter kernels in front of and behind a sparse merge took 18 + 21 us.  Workgroups
// of k_wide_scatter that do nothing else cost that kernel the 17 us they save this one).
template <typename I, typename S, typename O, bool DENSE>
__global__ __launch_bounds__(kWideBlock) void k_wide_merge(WideList list, I *__restrict__ out_idx,
                                                           O *__restrict__ out_val, int64_t capacity,
                                                           ScanState st, int tie_bits, int64_t *out_count,
                                                           HostAnswer answer) {
  __shared__ WideMergeShared sh;
  const SlabGeom &geo = list.geo;
  const WideSlabs &in = list.out;
  const uint32_t dense_n = list.dense_n;
  int32_t *const status = list.status;
  const uint32_t tid = threadIdx.x;
  if (tid == 0) {
    sh.tile = (int)atomicAdd(st.ticket, 1u);
    sh.qn = sh.big = 0;
  }
  sh.cnt.clear();
  __syncthreads();
  const uint32_t b = (uint32_t)__builtin_amdgcn_readfirstlane(sh.tile);  // buckets are taken in order, so every earlier bucket already runs
  const uint32_t nb = geo.nbuckets;
  if (b >= nb) return;
  const uint32_t lo = geo.first_key(b);
  // The bucket's range of a dense tensor: elements up to the first multiple of 16 bytes, vectors, elements.  The
  // vectors' zeros are stored a few at a time between the steps of the ranking loops, whose LDS round trips leave the
  // memory idle.
  constexpr uint32_t V = 16 / sizeof(O);
  uint32_t zero_vecs = 0, zero_at = tid, zero_each = 0;
  u32x4 *zero_to = nullptr;
  if (DENSE) {
    const uint32_t end = b + 1 < nb ? geo.first_key(b + 1) : dense_n;
    const uint32_t skew = (uint32_t)((reinterpret_cast<uintptr_t>(out_val + lo) & 15u) / sizeof(O));
    uint32_t head = (V - skew) % V;
    if (head > end - lo) head = end - lo;
    zero_vecs = (end - lo - head) / V;
    zero_to = reinterpret_cast<u32x4 *>(out_val + lo + head);
    for (uint32_t i = tid; i < head; i += kWideBlock) out_val[lo + i] = O(0);
    for (uint32_t i = lo + head + zero_vecs * V + tid; i < end; i += kWideBlock) out_val[i] = O(0);
  }
  auto zero_some = [&]() {
    if (!DENSE) return;
    const u32x4 zero = {0, 0, 0, 0};
    for (uint32_t i = 0; i < zero_each && zero_at < zero_vecs; ++i, zero_at += kWideBlock) zero_to[zero_at] = zero;
  };
  uint32_t pcount[kWideSplit];
  uint32_t longest = 0;
#pragma unroll
  for (int q = 0; q < kWideSplit; ++q) {
    pcount[q] = in.cursor[coarse_cursor_at(b, q)];
    if (pcount[q] > in.part_cap) pcount[q] = in.part_cap;  // the scatter flagged the overflow
    longest = pcount[q] > longest ? pcount[q] : longest;
  }
  if (DENSE) {  // two pauses in every step
    const uint32_t pauses = (longest <= (uint32_t)kWideBlock ? 1u : longest <= 2u * kWideBlock ? 2u : (uint32_t)kWmRounds) * (2u * kWideSplit / kWmLanes);
    zero_each = (zero_vecs + kWideBlock * pauses - 1u) / (kWideBlock * pauses);
  }
  bool declined = false;
  if (longest > (uint32_t)kWmPartMax) {
    declined = true;
#pragma unroll
    for (int q = 0; q < kWideSplit; ++q) pcount[q] = 0;
    longest = 0;
  }
  const uint32_t n =
      longest <= (uint32_t)kWideBlock ? wide_merge_sort<S, 1>(sh, geo, in, b, pcount, longest, declined, tie_bits, status, zero_some)
      : longest <= 2u * kWideBlock ? wide_merge_sort<S, 2>(sh, geo, in, b, pcount, longest, declined, tie_bits, status, zero_some)
                                   : wide_merge_sort<S, kWmRounds>(sh, geo, in, b, pcount, longest, declined, tie_bits, status, zero_some);
  // where this bucket's output starts: the sum of what all earlier buckets keep.  Every thread asks for one of
  // them (bounded wait), nobody waits for a chain of prefixes; while the answers are on their way the kept
  // entries are gathered in LDS.
  uint64_t d = kDescAggregate;
  auto publish = [&](uint32_t kept) {
    if (DENSE) return;
    if (tid == 0) desc_store(&st.desc[b], kDescAggregate | kept);
    if (tid < b) d = desc_load(&st.desc[tid]);
  };
  // written out for a few numbers of places a thread
  static_assert(kWmSumItems == 17, "as many as a full bucket needs");
  const uint32_t total = n <= 5u * kWideBlock    ? wide_merge_sums<O, DENSE, 5>(sh, n, lo, publish)
                         : n <= 9u * kWideBlock  ? wide_merge_sums<O, DENSE, 9>(sh, n, lo, publish)
                         : n <= 13u * kWideBlock ? wide_merge_sums<O, DENSE, 13>(sh, n, lo, publish)
                                                 : wide_merge_sums<O, DENSE, kWmSumItems>(sh, n, lo, publish);
  {
    uint32_t spins = 0;
    while ((d >> 62) == 0) {
      if (++spins > kSpinLimit) {
        atomicOr(status, ZEN_STAT_INTERNAL);
        break;
      }
      __builtin_amdgcn_s_sleep(2);
      d = desc_load(&st.desc[tid]);
    }
  }
  if (DENSE) {
    __syncthreads();  // the gathered entries are there
    for (uint32_t i = tid; i < total; i += kWideBlock) out_val[sh.key[i]] = SumAs<O>::of(sh.val[i]);
  } else {
    uint32_t all_before;  // (fewer than 2^31 entries in all)
    block_exclusive_scan<uint32_t, kWideBlock>((uint32_t)d, sh.scan, &all_before);  // its barriers also publish the gathered entries
    if (b == nb - 1 && tid == 0) {
      const uint64_t all = (uint64_t)all_before + total;
      // (for the launch's last workgroup to read, on another die maybe)
      __hip_atomic_store(out_count, (int64_t)all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (all > (uint64_t)capacity) atomicOr(status, ZEN_STAT_CAPACITY);
    }
    const uint64_t room = (uint64_t)capacity > all_before ? (uint64_t)capacity - all_before : 0;
    const uint32_t fits = total < room ? total : (uint32_t)room;
    I *const to_idx = out_idx + all_before;
    O *const to_val = out_val + all_before;
    for (uint32_t i = tid; i < fits; i += kWideBlock) {
      to_idx[i] = (I)sh.key[i];
      to_val[i] = SumAs<O>::of(sh.val[i]);
    }
  }
  if (answer.host) wait_global_acks();  // its share of the status word, and the count
  // every workgroup has read the descriptors it needs before it gets here: the last one to finish clears the
  // prefix state
  __syncthreads();
  if (tid == 0) sh.tile = done_last(list.done, b, nb);
  __syncthreads();
  if (sh.tile) {
    for (uint32_t i = tid; i < nb; i += kWideBlock) st.desc[i] = 0ull;
    if (tid < kDoneWords) list.done[tid] = 0;
    if (tid == 0) *st.ticket = 0;
    host_answer_count(answer, DENSE ? nullptr : out_count, status);
  }
}

}  // namespace

bool wide_merge_fits(int64_t r, int64_t dense_n, int cus, SlabGeom *geo, bool alone) {
  SlabGeom g;
  // (shorter lists: one workgroup, zen_merge.hip)
  if (r <= merge_one_max() || r > 0x7ffffffell || cus <= 0) return false;
  // Sixteen buckets for small index ranges, more only for lists that need them: a bucket's workgroup takes a compute
  // unit, and 128 of them for ten thousand entries keep the encode beside them waiting (a step of 1 Mi elements
  // took 106 us instead of 85).
  const int64_t least = ceil_div(r, (int64_t)8192) > 16 ? ceil_div(r, (int64_t)8192) : 16;
  int64_t width = dense_n / least < 4ll * kWideSubs ? dense_n / least : 4ll * kWideSubs;
  if (width < 1024) width = 1024;
  if (!wide_geometry(dense_n, 1, r, cus, &g, 1ll << 14, width, alone)) return false;
  if (g.sub_shift + ceil_log2_u64((uint64_t)r) > 32) return false;  // (index inside a narrow range, arrival number) must fit a word
  // a slab record carries the index's offset inside its bucket and the arrival number in fixed fields
  if ((uint64_t)g.sub_shift + 14 > kWmOffBits || (uint64_t)r >= (1ull << kWmArrBits)) return false;
  if (geo) *geo = g;
  return true;
}

static uint32_t wide_merge_part_cap(const SlabGeom &geo, int64_t r) { return wide_part_cap(geo, r + r / 4); }

// Workspace of the wide path behind the zero region at the head of zen_merge's workspace.
size_t wide_merge_bytes(int64_t r, int64_t dense_n, int cus) {
  size_t entries = 0;
  for (const bool alone : {false, true}) {
    SlabGeom geo;
    if (!wide_merge_fits(r, dense_n, cus, &geo, alone)) continue;
    const size_t e = (size_t)geo.nbuckets * kWideSplit * wide_merge_part_cap(geo, r);
    if (e > entries) entries = e;
  }
  if (!entries) return 0;
  return align_up(entries * sizeof(uint2), 256) + align_up(entries * sizeof(uint32_t), 256);
}

// The received entries as the scatter wants them: cursor: kCoarseCursorWords zeroed words (zero again when
// k_wide_merge has run); done: kDoneWords of the same kind; rest: wide_merge_bytes(...) bytes.  False if the sizes do not suit the wide buckets.
bool wide_merge_list(const void *idx, int idx64_in, const void *val, int64_t r, int64_t dense_n, uint32_t *cursor,
                     uint32_t *done, void *rest, int cus, int32_t *status, WideList *list, bool alone) {
  SlabGeom geo;
  if (!wide_merge_fits(r, dense_n, cus, &geo, alone)) return false;
  WideSlabs slabs;
  slabs.part_cap = wide_merge_part_cap(geo, r);
  const size_t entries = (size_t)geo.nbuckets * kWideSplit * slabs.part_cap;
  Carver cv(rest);
  slabs.cursor = cursor;
  slabs.rec = cv.take<uint2>(entries);
  slabs.val32 = cv.take<uint32_t>(entries);
  list->geo = geo;
  list->idx = idx;
  list->val = val;
  list->r = (uint32_t)r;
  list->dense_n = (uint32_t)dense_n;
  list->idx64 = idx64_in;
  list->out = slabs;
  list->done = done;
  list->status = status;
  return true;
}

uint32_t wide_scatter_batches(const WideList &list, int batch) { return (uint32_t)ceil_div((int64_t)list.r, batch); }

template <typename S, typename O>
static void wide_merge_launch(const WideList &list, void *out_idx, int idx64_out, O *out_val, int64_t capacity,
                              int64_t *out_count, unsigned long long *scan, hipStream_t s, const HostAsk &ask) {
  const ScanState st = scan_state(scan, (int64_t)list.geo.nbuckets);
  const int tie_bits = ceil_log2_u64((uint64_t)list.r);  // arrival numbers are < r
  const dim3 grid(list.geo.nbuckets), block(kWideBlock);
  if (!out_idx)
    k_wide_merge<int32_t, S, O, true><<<grid, block, 0, s>>>(list, nullptr, out_val, capacity, st, tie_bits, out_count,
                                                                         ask.answer);
  else if (idx64_out)
    k_wide_merge<int64_t, S, O, false><<<grid, block, 0, s>>>(list, static_cast<int64_t *>(out_idx), out_val, capacity,
                                                                     st, tie_bits, out_count, ask.answer);
  else
    k_wide_merge<int32_t, S, O, false><<<grid, block, 0, s>>>(list, static_cast<int32_t *>(out_idx), out_val, capacity,
                                                                     st, tie_bits, out_count, ask.answer);
}

static void wide_merge_typed(const WideList &list, int dtype, void *out_idx, int idx64_out, void *out_val, int out_dtype,
                             int64_t capacity, int64_t *out_count, unsigned long long *scan, hipStream_t s,
                             const HostAsk &ask) {
  if (dtype == ZEN_F32)
    wide_merge_launch<uint32_t, float>(list, out_idx, idx64_out, static_cast<float *>(out_val), capacity, out_count, scan, s, ask);
  else if (out_dtype == ZEN_BF16)
    wide_merge_launch<uint16_t, uint16_t>(list, out_idx, idx64_out, static_cast<uint16_t *>(out_val), capacity, out_count, scan, s, ask);
  else
    wide_merge_launch<uint16_t, float>(list, out_idx, idx64_out, static_cast<float *>(out_val), capacity, out_count, scan, s, ask);
}

// The two launches.  scan: zeroed prefix state for 256 buckets (descriptors, ticket), zero again
// when the second ends.  out_dtype: ZEN_F32 (the sums; the only choice for fp32 values) or ZEN_BF16 (rounded).
// out_idx == nullptr: out_val is the dense tensor.
int wide_merge(const WideList &list, int dtype, void *out_idx, int idx64_out, void *out_val, int out_dtype,
               int64_t capacity, int64_t *out_count, unsigned long long *scan, hipStream_t s, const HostAsk &ask) {
  {
    ProfScope prof(kProfWideScatter, s);
    if (dtype == ZEN_BF16)
      k_wide_scatter<uint16_t><<<dim3(wide_scatter_batches(list, kWsBatch)), dim3(kWsBlock), 0, s>>>(list);
    else
      k_wide_scatter<uint32_t><<<dim3(wide_scatter_batches(list, kWsBatch)), dim3(kWsBlock), 0, s>>>(list);
    ZEN_LAUNCH_CHECK("k_wide_scatter");
  }
  ProfScope prof(kProfWideMerge, s);
  wide_merge_typed(list, dtype, out_idx, idx64_out, out_val, out_dtype, capacity, out_count, scan, s, ask);
  ZEN_LAUNCH_CHECK("k_wide_merge");
  if (ask.answer.host) *ask.answered = true;
  return ZEN_OK;
}

}  // namespace zen
