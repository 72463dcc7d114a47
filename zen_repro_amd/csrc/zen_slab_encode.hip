// Fused load balance on bucket slabs (the fast path of zen_load_balance).
//
// The reference inserts every selected index into an int32 table as large as
// the gradient and then scans that table partition by partition
// (functions_cuda_kernel.cu:97-167, tensor_load_balance.py:13-51).  Here the
// select kernel leaves its candidates in 64 coarse slabs (a coarse slab = the
// level-1 hash slots of a group of buckets; a bucket is a range of level-1
// slots, zen_slab.h), and four or five short kernels finish the job:
//   k_fine_scatter  the coarse slabs, filtered by the exact threshold, go to the
//                   bucket slabs, so that every store belongs to a long run;
//   k_slab_sort     one workgroup per bucket: puts the bucket in the order of its
//                   level-1 slots by a bitmap of them in LDS (wide buckets: by
//                   comparing entries); of the entries that share a slot the one
//                   with the smallest index is its level-1 owner, the others lost
//                   level 1;
//   k_slab_settle   (where many losers are expected) their level-2 slots, a group
//                   of buckets at a time in LDS;
//   k_slab_chains   levels 2 and 3 for the losers that are left through a small
//                   hash map, with the reference's rule executed in ascending
//                   index order (a slot belongs to the smallest index that ever
//                   probes it; whoever takes a slot from a larger index continues
//                   that index's probe sequence).  Every bucket has a part of the
//                   map of its own, so what finally moved into a bucket is what
//                   its part holds; an index that ran out of levels goes to its
//                   partition's serial list; split sizes;
//   k_slab_place    one workgroup per bucket: survivors and moved-in entries by
//                   the same kind of bitmap to the bucket's place in the
//                   partition-major output.
#include <algorithm>

#include "zen_balance.h"
#include "zen_hashmap.h"
#include "zen_slab.h"
#include "zen_slab_feed.h"
#include "zen_refine.h"

namespace zen {
namespace {

struct SlabTables {
  uint32_t *cursor;     // [B] records in the bucket's slab
  uint32_t *bucket_lo;  // [B] smallest level-1 slot of the bucket
  uint32_t *bucket_n;   // [B] sorted records in the slab: level-1 owners, in wide buckets the losers too
  uint32_t *removed_n;  // [B] of which have lost their slot
  uint32_t *movein_n;   // [B * kMoveinPad] occupied cells of the bucket's part of the map: entries that moved in
  uint32_t *serial_n;   // [P * kMoveinPad] entries that found no slot
  uint32_t *raw_idx;    // [B * kSlabCap] entries as they arrive: index (after the sort: losers, again_n of them) ...
  void *raw_val;        // ... and value
  int32_t *slab_idx;    // [B * kSlabCap] after the sort: index | kRemovedBit, by ascending level-1 slot (the slot
                        // itself is not kept: hashing the index again is cheaper than a trip to memory)
  void *slab_val;       // [B * kSlabCap] after the sort: value
  uint16_t *sub_index;  // [B * kSlabIndexLen] sorted place of the first record of every kSlabIndexStep-th narrow
                        // key range of the bucket (the last entry: the number of records)
  uint32_t *ser_idx;    // [P * kSlabSerialCap]
  uint32_t *again_n;    // [B] losers the bucket's sort found, but for those in the groups' lists
  uint32_t *group_n;    // [P * group_pad] losers whose level-2 slot is one of the group's ...
  uint32_t *group_list; // [groups * group_cap] ... and who they are
  uint32_t *token_n;    // [groups] indices that k_slab_settle leaves to k_slab_chains ...
  uint32_t *token;      // [groups * group_cap] ... and who they are (kAtLevel3: at which level)
  uint32_t *out_start;  // [B + 1] where every bucket starts in the output
  uint32_t *done;       // [kDoneWords] workgroups of k_slab_chains that have finished
  uint32_t *final_n;    // [B + P] what k_slab_place needs of the counters above, copied by the last workgroup of
                        // k_slab_chains before it puts them back to zero: moved-in entries per bucket, serial entries
                        // per partition
  uint32_t *coarse_cursor;  // the feed's coarse cursors and, for an fp32 top-k, the refinement histogram (else
  uint32_t *refine_hist;    // null): k_slab_sort puts them back to zero
  int partitions;
  uint32_t gpp;         // groups in a partition ...
  uint32_t per_group;   // ... of so many buckets
  uint32_t group_pad;   // words from one partition's counters to the next's
  uint32_t group_cap;   // losers in a group's list (0: no lists), at most kSettleRows to a thread of its workgroup
};

// Device-wide atomics on one 128-byte line are carried out one after the other: four counters to a line.
constexpr uint32_t kMoveinPad = 8;

// A cell of the map: (slot + 1) << 32 | index, 0 if empty.
__device__ inline uint32_t cell_slot(unsigned long long cell) { return (uint32_t)(cell >> 32) - 1u; }

// Where many losers are expected a bucket's losers go to lists, by the group of buckets their level-2 slots lie in, and
// k_slab_settle enters a group's list into its parts of the map in LDS: device-wide atomics are carried out at 25 a
// nanosecond, and of an entry for each loser in the map and one to count it nine in ten fall away.  Where fewer are
// expected each goes its way through memory (k_slab_chains), for the other way is a launch more and two barriers in the sort.
// What settling costs goes with the buckets, what it saves with the losers.  Whole calls, bf16, 62 M slots, sixteen partitions,
// by expected losers to a bucket, unsettled and settled, us: with a capacity of 1.05 times what is selected 120 115.2 and 114.5,
// 146 122.9 and 122.8, 195 127.0 and 123.4, 244 142.2 and 134.7, 325 202.9 and 180.3, 382 313.8 and 255.5; with 1.5 times, of
// whose losers fewer than a half come, 239 43.5 and 45.3 (sort, settling and chains).  The line lies between the two.  62 M, an odd
// number: 105 118.4 and 120.9, 174 131.7 and 130.3, 206 203.5 and 188.3.  2^26: 129 122.7 and 123.4, 232 149.0 and 146.5; 2^28:
// 120 307.1 and 314.6.  Few in all, 4 to 17 M slots: 29 000 55.6 and 54.9, 55.7 and 56.8, 59.9 and 60.6; 44 000 62.8 and 61.3, 61.7
// and 60.1; 59 000 69.6 and 65.5, 74.7 and 74.5.  Many in all, 250 M slots, 3072 and 3584 buckets: 440 000 300.4 and 294.2,
// 549 000 347.5 and 328.9.
constexpr double kSettleFrom = 250, kSettleLeast = 50000, kSettleAnyway = 400000;
constexpr uint32_t kGroupBuckets = 12;         // of a group, at most: their parts of the map and indices fill 121 KB
constexpr uint32_t kGroupLeast = 4, kGroupsMost = 256;  // (a compute unit to each)
constexpr uint32_t kMostGroups = kSlabMaxBuckets / kGroupBuckets + 1;  // of a partition
constexpr int kSettleBlock = 1024;
constexpr int kSettleRows = 6;                 // losers of a thread, at most
// More partitions than kGroupsMost: groups of a few buckets, five to a compute unit.  62 M slots, by expected losers to a bucket:
// 300 partitions 99 105.9 and 106.7 us, 159 138.4 and 133.6, 199 157.9 and 147.4, 408 294 and 245; 700: 142 126.7 and 127.8,
// 171 139.8 and 138.0; 1300: 153 139.0 and 134.2; 3000: 99 176 and 179, 166 226 and 213, 326 324 and 271.  (The line leaves room
// for larger capacities here too.)
constexpr double kSettleFewFrom = 190;
constexpr uint32_t kFewBuckets = 3, kFewGroupsMost = 1280;
constexpr int kFewBlock = 256;
constexpr uint32_t kChainsResident = 1024;     // workgroups of k_slab_chains the chip holds at a time
constexpr uint32_t kAtLevel3 = 1u << 31;       // in a list: the index goes on at level 3 (else at level 2)

// The counters and histograms that must be zero when a call starts live in memory that is zero between calls
// (the part of the caller's table the hash map does not use), and every one of them is put back to zero by the
// last kernel that needs it: no kernel spends its time clearing them up front.

// Every kSlabIndexStep-th narrow key range of a bucket (zen_slab.h; about one record per range) has its first
// sorted place written down by the sort kernel: whoever asks who owns a level-1 slot reads two of these places
// and the three or four records between them instead of bisecting the whole bucket (thirteen loads, one
// after the other).
constexpr int kSlabIndexStep = 4;
constexpr int kSlabIndexLen = kSlabSubs / kSlabIndexStep + 1;
static_assert(kSlabSubs % kSlabIndexStep == 0 && kSlabCap < 65536, "index layout");

// ---------------------------------------------- coarse slabs -> bucket slabs

// The select kernel leaves its candidates in the coarse slabs (zen_slab_feed.h), as (index, value): index 0 is
// dropped there already, what the exact threshold excludes is dropped on the way to the buckets (the threshold
// is known only when the select kernel has ended).  An entry's level-1 slot is hashed again wherever it is
// needed, which is cheaper than carrying it along.
template <typename S>
struct EncodeSink {
  SlabGeom geo;
  uint32_t *raw_idx;
  S *raw_val;
  const uint32_t *filter;  // optional exact threshold
  __device__ inline bool keep(const uint32_t (&w)[2]) const {
    return (w[1] & KeyOf<S>::kMask) >= (filter ? filter[0] : 0u);
  }
  __device__ inline uint32_t bucket(const uint32_t (&w)[2]) const {
    return geo.bucket_of(geo.mod_m(poly(w[0]) + kSeed1));
  }
  __device__ inline void store(size_t at, const uint32_t (&w)[2]) const {
    raw_idx[at] = w[0];
    raw_val[at] = (S)w[1];
  }
};

// ------------------------------------------------------------ sort a bucket

// Two ways to put a bucket in order.  By a bitmap of its slots (k_slab_sort, k_slab_place) the work goes with the slots:
// these kernels come in two widths, with which two workgroups share a compute unit.  By comparing records
// (k_slab_sort_wide, k_slab_place_wide) it goes with the records, whatever the width.  A bucket within the second width
// takes the bitmap.  Where the buckets the records call for are wider, more of them are made for the bitmap's sake up
// to kSlabSparse slots per record of the capacity.  bf16, sort + place + chains, bitmap and comparisons: 2^30 slots,
// 10.7 M records 116 us and (at the time, the bitmap 127) 170, 7.5 M 104 and 104, 6.4 M 94 and 92, 5.4 M 91 and 78; 1 M on
// 1024 partitions 87 and 40.  No number of buckets makes the widest tables fit (more than 1.34 G slots): a bitmap of nine
// 2^16 slots, one workgroup to a compute unit, took 216 us for 1.34 G slots and 6.7 M records, comparisons 106 (99 now);
// 2.1 G slots and 4.3 M records 216 and 75.
constexpr uint32_t kSlabSpan1 = 1u << 17, kSlabSpan2 = 5u << 16;
constexpr int64_t kSlabSparse = 128;

constexpr int kSortBlock = 1024;
constexpr int kSortItems = kSlabCap / kSortBlock;

template <typename S, uint32_t SPAN>
struct SlabSortLds {
  uint32_t idx[kSlabCap];  // the sorted indices
  union {
    SlabTaken<SPAN> taken;
    struct {               // once the ranks are known:
      S val[kSlabCap];         // the sorted values
      uint32_t list[kSlabCap]; // the losers
    };
  };
  uint32_t scan[kSortBlock / 64 + 1];
  uint32_t shared, lost, again;
};

// Sorts a bucket's records by level-1 slot; of those that share a slot the smallest index owns it, the others are
// listed and not kept.  A bucket has a few to a few hundred slots per record, so the slots are marked in a bitmap: a
// record's place is the number of marks below its own, and whoever finds its slot marked already is settled by the
// smallest index afterwards.  Bound by the vector instructions and the LDS round trips behind every phase's barrier (two
// workgroups a compute unit).  ROWS: records of a thread (the last row may be cut short); the code is written out for
// each number, so that all marks and all look-ups of a phase are on their way together (with one body for all numbers
// and branches around the rows a wave waited for every single mark): 62 M slots, 6.2 M bf16 records 46 -> 42 us, 3.1 M
// 23.7 -> 21.5.  (By comparisons, k_slab_sort_wide: 64 and 33 at the time.)
template <int ROWS, typename S, uint32_t SPAN>
__device__ __forceinline__ void slab_sort_rows(SlabSortLds<S, SPAN> &sh, const SlabGeom &geo, const SlabTables &tb,
                                               uint32_t n_raw) {
  const uint32_t b = blockIdx.x;
  const size_t base = (size_t)b * kSlabCap;
  const uint32_t words = (geo.span + 63u) / 64u;
  const uint32_t lo = tb.bucket_lo[b];
  const char *raw_idx = reinterpret_cast<const char *>(tb.raw_idx + base);
  const char *raw_val = reinterpret_cast<const char *>(static_cast<const S *>(tb.raw_val) + base);
  uint32_t off[ROWS], idx[ROWS], rank[ROWS];
  S val[ROWS];
  uint32_t live = 0, owner = 0;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const uint32_t j = threadIdx.x + i * kSortBlock;
    // no branch around a wave's loads (places past the end are pulled back onto the slab's first record): they are
    // all in flight together
    const uint32_t from = j < n_raw ? j : 0u;
    idx[i] = *reinterpret_cast<const uint32_t *>(raw_idx + (uint32_t)(from * sizeof(uint32_t)));
    val[i] = *reinterpret_cast<const S *>(raw_val + (uint32_t)(from * sizeof(S)));
    live |= (j < n_raw ? 1u : 0u) << i;
  }
  __syncthreads();  // the bitmap is clear, and everybody has read the slab's fill count
  if (threadIdx.x == 0) tb.cursor[b] = 0;
  // no branch around a wave's marks either: a lane without a record marks nothing
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    off[i] = geo.mod_m(poly(idx[i]) + kSeed1) - lo;  // the level-1 slot again: cheaper than carrying it along
    if (!(live & (1u << i))) off[i] = 0;
    rank[i] = sh.taken.take(off[i], (live >> i) & 1u);
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) owner |= (~(rank[i] >> (off[i] & 31u)) & 1u) << i;  // the first to mark its slot
  owner &= live;
  if (owner != live) sh.shared = 1;
  __syncthreads();
  const uint32_t n = sh.taken.template count<kSortBlock>(words, sh.scan);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ROWS; ++i) rank[i] = sh.taken.place(off[i]);
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    if (owner & (1u << i)) sh.idx[rank[i]] = idx[i];
  // every kSlabIndexStep-th narrow range's first sorted place goes to the index
  for (int j = threadIdx.x; j < kSlabIndexLen; j += kSortBlock) {
    const uint32_t first = (uint32_t)j * kSlabIndexStep << geo.sub_shift;
    tb.sub_index[(size_t)b * kSlabIndexLen + j] = (uint16_t)(first < geo.span ? sh.taken.place(first) : n);
  }
  __syncthreads();
  if (sh.shared) {  // (the same for the whole workgroup)
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      if ((live & ~owner) & (1u << i)) atomicMin(&sh.idx[rank[i]], idx[i]);
    __syncthreads();
    uint32_t own[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) own[i] = sh.idx[rank[i]];
    owner = 0;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) owner |= (own[i] == idx[i] ? 1u : 0u) << i;
    owner &= live;
  }
  const uint32_t losers = live & ~owner;
  uint32_t at = losers ? atomicAdd(&sh.lost, (uint32_t)__popc(losers)) : 0u;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    if (owner & (1u << i)) sh.val[rank[i]] = val[i];  // (the bitmap has done its work)
    if (losers & (1u << i)) sh.list[at++] = idx[i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    tb.bucket_n[b] = n;
    tb.removed_n[b] = 0;
  }
  int32_t *slab_idx = tb.slab_idx + base;
  S *slab_val = static_cast<S *>(tb.slab_val) + base;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const uint32_t p = threadIdx.x + i * kSortBlock;
    if (p < n) {
      slab_idx[p] = (int32_t)sh.idx[p];
      slab_val[p] = sh.val[p];
    }
  }
}

// LISTS: the losers go to the groups' lists (a kernel of its own: beside the merge's workgroups the other one gets along
// better without that code).
template <typename S, uint32_t SPAN, bool LISTS>
__global__ __launch_bounds__(kSortBlock, 8) void k_slab_sort(SlabGeom geo, SlabTables tb) {
  __shared__ SlabSortLds<S, SPAN> sh;
  const uint32_t b = blockIdx.x;
  const uint32_t words = (geo.span + 63u) / 64u;
  uint32_t n_raw = tb.cursor[b];
  if (n_raw > (uint32_t)kSlabCap) n_raw = kSlabCap;  // the scatter flagged the overflow
  if (threadIdx.x == 0) sh.shared = sh.lost = sh.again = 0;
  sh.taken.template clear<kSortBlock>(words);
  // the kernels before this one were the last to need these: back to zero, a slice per workgroup
  for (uint32_t i = b * kSortBlock + threadIdx.x; i < kCoarseCursorWords; i += gridDim.x * kSortBlock)
    tb.coarse_cursor[i] = 0;
  if (tb.refine_hist)
    for (uint32_t i = b * kSortBlock + threadIdx.x; i < (uint32_t)kRefineWords; i += gridDim.x * kSortBlock)
      tb.refine_hist[i] = 0;
  static_assert(kSortItems == 6, "a case for every number of rows");
  switch ((n_raw + kSortBlock - 1) / kSortBlock) {
    case 0:
    case 1: slab_sort_rows<1>(sh, geo, tb, n_raw); break;
    case 2: slab_sort_rows<2>(sh, geo, tb, n_raw); break;
    case 3: slab_sort_rows<3>(sh, geo, tb, n_raw); break;
    case 4: slab_sort_rows<4>(sh, geo, tb, n_raw); break;
    case 5: slab_sort_rows<5>(sh, geo, tb, n_raw); break;
    default: slab_sort_rows<6>(sh, geo, tb, n_raw); break;
  }
  // The losers, to the groups' lists a run of each (one atomic to a group), else to the bucket's own: that is the memory of
  // the records' indices, which have been in registers since the first barrier.  (One log for all buckets, and its one
  // counter, 11 ns a workgroup: 268 M slots, 2.7 M bf16 records in 1024 buckets 22.2 us, so 19.3.)
  uint32_t *own = tb.raw_idx + (size_t)b * kSlabCap;
  if constexpr (!LISTS) {
    for (uint32_t i = threadIdx.x; i < sh.lost; i += kSortBlock) own[i] = sh.list[i];
    if (threadIdx.x == 0) tb.again_n[b] = sh.lost;
    return;
  }
  const uint32_t part = b / geo.bpp;
  uint32_t *count = sh.idx;  // of every group (the sorted indices are on their way out)
  static_assert(kMostGroups <= kSlabCap && kMostGroups <= kSortBlock, "a group per thread");
  for (uint32_t i0 = 0; i0 < sh.lost; i0 += kSortBlock) {  // (one turn as a rule)
    __syncthreads();
    if (threadIdx.x < tb.gpp) count[threadIdx.x] = 0;
    __syncthreads();
    const bool one = i0 + threadIdx.x < sh.lost;
    uint32_t t = 0, to = 0, at = 0;
    if (one) {
      t = sh.list[i0 + threadIdx.x];
      to = (geo.spot(t, 1).bucket - part * geo.bpp) / tb.per_group;
      at = atomicAdd(&count[to], 1u);
    }
    __syncthreads();
    if (threadIdx.x < tb.gpp) {
      const uint32_t n = count[threadIdx.x];
      if (n) count[threadIdx.x] = atomicAdd(&tb.group_n[part * tb.group_pad + threadIdx.x], n);
    }
    __syncthreads();
    if (one) {
      at += count[to];
      if (at < tb.group_cap)
        tb.group_list[(size_t)(part * tb.gpp + to) * tb.group_cap + at] = t;
      else
        own[atomicAdd(&sh.again, 1u)] = t;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) tb.again_n[b] = sh.again;
}

// The same for few records among many slots: grouped by narrow key ranges, ranked against the words of their group
// (slab_rank), the owners found by walking the sorted runs.  Those that lost stay where they are, marked.  Bound by LDS
// round trips: 1.48 G slots, 14.7 M bf16 records 98 us; 1.34 G and 6.7 M 50.
template <typename S>
__global__ __launch_bounds__(kSortBlock, 8) void k_slab_sort_wide(SlabGeom geo, SlabTables tb, int32_t *status) {
  // the ties take the place of the counters once the ranks are known: with 32-bit values the kernel would
  // otherwise need 88 KB of LDS, one workgroup to a compute unit instead of two
  __shared__ SlabSortSharedNoQueue sh;
  __shared__ S s_val[kSlabCap];
  __shared__ uint32_t s_lost;
  const uint32_t b = blockIdx.x;
  const size_t base = (size_t)b * kSlabCap;
  uint32_t n_raw = tb.cursor[b];
  if (n_raw > (uint32_t)kSlabCap) n_raw = kSlabCap;  // the scatter flagged the overflow
  const uint32_t lo = tb.bucket_lo[b];
  S *slab_val = static_cast<S *>(tb.slab_val);
  if (threadIdx.x == 0) s_lost = 0;
  // the kernels before this one were the last to need these: back to zero, a slice per workgroup
  for (uint32_t i = b * kSortBlock + threadIdx.x; i < kCoarseCursorWords; i += gridDim.x * kSortBlock)
    tb.coarse_cursor[i] = 0;
  if (tb.refine_hist)
    for (uint32_t i = b * kSortBlock + threadIdx.x; i < (uint32_t)kRefineWords; i += gridDim.x * kSortBlock)
      tb.refine_hist[i] = 0;
  uint32_t off[kSortItems], idx[kSortItems], pos[kSortItems], rank[kSortItems];
  S val[kSortItems];
  uint32_t live = 0;
#pragma unroll
  for (int i = 0; i < kSortItems; ++i) {
    const uint32_t j = threadIdx.x + i * kSortBlock;
    // no branch around the loads (places past the end are pulled back onto the slab's first record): they are
    // all in flight together
    const size_t from = base + (j < n_raw ? j : 0u);
    idx[i] = tb.raw_idx[from];
    val[i] = static_cast<const S *>(tb.raw_val)[from];
    off[i] = pos[i] = 0;
    if (j < n_raw) {
      off[i] = geo.mod_m(poly(idx[i]) + kSeed1) - lo;  // the level-1 slot again: cheaper than carrying it along
      pos[i] = j;
      live |= 1u << i;
    }
  }
  // ties between equal slots are broken by the record's place in the slab (13 bits, so a record is one word
  // while it is ranked); the runs of equal slots, few and short, are put right afterwards
  static_assert(kSlabCap <= (1 << 13), "slab places in 13 bits");
  uint32_t n = 0;
  if (!slab_rank<kSortBlock>(sh, geo, 13, off, pos, live, rank, &n)) {
    if (threadIdx.x == 0) {
      tb.cursor[b] = 0;
      atomicOr(status, ZEN_STAT_RETRY);
      tb.bucket_n[b] = 0;
      tb.removed_n[b] = 0;
      tb.again_n[b] = 0;
    }
    for (int j = threadIdx.x; j < kSlabIndexLen; j += kSortBlock) tb.sub_index[(size_t)b * kSlabIndexLen + j] = 0;
    return;
  }
  // every thread has read the slab's fill count (slab_rank synchronised); this workgroup was its only reader
  if (threadIdx.x == 0) tb.cursor[b] = 0;
  // the counters hold where every narrow range starts in the sorted bucket: every kSlabIndexStep-th goes to
  // the index (before the counters' memory is used for the ties below)
  for (int j = threadIdx.x; j < kSlabIndexLen; j += kSortBlock)
    tb.sub_index[(size_t)b * kSlabIndexLen + j] = (uint16_t)sh.cnt[j * kSlabIndexStep];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSortItems; ++i) {
    if (live & (1u << i)) {
      sh.key[rank[i]] = off[i];
      sh.tie[rank[i]] = idx[i];
      s_val[rank[i]] = val[i];
    }
  }
  __syncthreads();
  // a run of equal slots gets its smallest index in front (the thread at the run's first place does it)
  for (uint32_t p = threadIdx.x; p + 1 < n; p += kSortBlock) {
    const uint32_t k = sh.key[p];
    if (sh.key[p + 1] == k && (p == 0 || sh.key[p - 1] != k)) {
      uint32_t best = p;
      for (uint32_t u = p + 1; u < n && sh.key[u] == k; ++u)
        if (sh.tie[u] < sh.tie[best]) best = u;
      if (best != p) {
        const uint32_t ti = sh.tie[p];
        const S tv = s_val[p];
        sh.tie[p] = sh.tie[best];
        s_val[p] = s_val[best];
        sh.tie[best] = ti;
        s_val[best] = tv;
      }
    }
  }
  __syncthreads();
  // In a run of equal slots the first entry has the smallest index: the slot's level-1 owner.  The others
  // lost level 1.  Their places in the sorted slab are collected where the slots were, once every thread has
  // looked at those (a bucket has at most kSlabSubs of them, else the call is declined).
  uint32_t lost_mask = 0;
#pragma unroll 1
  for (int i = 0; i < kSortItems; ++i) {
    const uint32_t p = threadIdx.x + (uint32_t)i * kSortBlock;
    if (p < n) {
      const uint32_t k = sh.key[p];
      const bool lost = p > 0 && sh.key[p - 1] == k;
      tb.slab_idx[base + p] = (int32_t)(sh.tie[p] | (lost ? kRemovedBit : 0u));
      slab_val[base + p] = s_val[p];  // every thread has read its records: in place is safe
      lost_mask |= lost ? 1u << i : 0u;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int i = 0; i < kSortItems; ++i) {
    if (lost_mask & (1u << i)) {
      const uint32_t at = atomicAdd(&s_lost, 1u);
      if (at < (uint32_t)kSlabSubs) sh.key[at] = threadIdx.x + (uint32_t)i * kSortBlock;
    }
  }
  __syncthreads();
  uint32_t lost_n = s_lost;
  if (lost_n > (uint32_t)kSlabSubs) {
    if (threadIdx.x == 0) atomicOr(status, ZEN_STAT_RETRY);
    lost_n = kSlabSubs;
  }
  for (uint32_t i = threadIdx.x; i < lost_n; i += kSortBlock) tb.raw_idx[base + i] = sh.tie[sh.key[i]];
  if (threadIdx.x == 0) {
    tb.bucket_n[b] = n;
    tb.removed_n[b] = lost_n;
    tb.again_n[b] = lost_n;
  }
}

// ------------------------------------------------------ levels 2 and 3

// Smallest index whose level-1 slot is `at.slot` (kNone if nobody's) and where it sits.  The bucket's index
// narrows the search to the records of kSlabIndexStep narrow ranges (three or four); they are fetched four at
// a time and looked at in sorted order: by ascending slot, and in a run of equal slots the smallest index
// comes first.
__device__ inline uint32_t slab_head(const SlabGeom &geo, const SlabTables &tb, const SlabGeom::Spot &at, size_t *pos_out) {
  const int32_t *idx = tb.slab_idx + (size_t)at.bucket * kSlabCap;
  const uint32_t j = (at.offset >> geo.sub_shift) / (uint32_t)kSlabIndexStep;
  const uint16_t *index = tb.sub_index + (size_t)at.bucket * kSlabIndexLen;
  uint16_t range[2];  // one load each time: a wave's lanes all read other lines
  __builtin_memcpy(range, index + j, sizeof(range));
  const uint32_t end = range[1];
  for (uint32_t p = range[0]; p < end; p += 4) {
    uint32_t t[4];  // (up to three words past the range are read and not looked at: the workspace goes on behind)
    __builtin_memcpy(t, idx + p, sizeof(t));
#pragma unroll
    for (int q = 0; q < 4; ++q) t[q] &= kIndexMask;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (p + q >= end) return kNone;
      const uint32_t s1 = geo.mod_m(poly(t[q]) + kSeed1);
      if (s1 > at.slot) return kNone;
      if (s1 == at.slot) {
        *pos_out = (size_t)at.bucket * kSlabCap + p + q;
        return t[q];
      }
    }
  }
  return kNone;
}

// Enters t as a prober of `slot` in bucket b's part of the map; returns the smallest earlier prober (kNone: there was
// none).  *full is set if the part has no room.
__device__ inline uint32_t part_min(unsigned long long *cells, uint32_t b, uint32_t slot, uint32_t t, bool *full) {
  unsigned long long *part = cells + ((size_t)b << kSlabPartLog2);
  constexpr uint32_t mask = (1u << kSlabPartLog2) - 1u;
  const unsigned long long mine = ((unsigned long long)(slot + 1u) << 32) | t;
  uint32_t h = cell_home(slot, kSlabPartLog2);
  for (uint32_t probes = 0; probes <= mask; ++probes, h = (h + 1u) & mask) {
    const unsigned long long cur = atomicCAS(&part[h], 0ull, mine);
    if (cur == 0ull) return kNone;
    if (cell_slot(cur) == slot) return (uint32_t)atomicMin(&part[h], mine);
  }
  *full = true;
  return 0u;  // pretend a smaller index owns it: the chain moves on and the call is retried anyway
}

// Where every bucket starts in the output: survivors + moved-in entries, the partition's serial entries
// behind its last bucket.  Run by one workgroup of kSlabBlock threads once all counts are final: it is the last
// to need the counters the chains raised with atomics, hands what k_slab_place still wants of them on in final_n
// and puts them back to zero.  What the status word can come to is known here too (k_slab_place adds nothing).
// The chip waits for this one workgroup: one trip to memory for all counts, by consecutive lanes, and prefixes in LDS
// (s_start: kSlabMaxBuckets + 1 words).  A thread with neighbouring buckets of its own asked for a memory line a lane: 2560
// buckets 9 us.
__device__ inline void slab_output_starts(const SlabGeom &geo, const SlabTables &tb, uint32_t *s_scan, uint32_t *s_start,
                                          int64_t spp, uint32_t capacity, int64_t *splits, const HostAnswer &answer,
                                          int32_t *status) {
  constexpr uint32_t kPer = kSlabMaxBuckets / kSlabBlock;
  const uint32_t B = geo.nbuckets, P = (uint32_t)tb.partitions;
  uint32_t mv[kPer], rm[kPer], n[kPer], sn[kPer];
#pragma unroll
  for (uint32_t e = 0; e < kPer; ++e) {  // (the conditions are the same for all threads: all loads are in flight together)
    const uint32_t x = threadIdx.x + e * (uint32_t)kSlabBlock;
    if (e * (uint32_t)kSlabBlock < B) {
      const uint32_t at = x < B ? x : 0u;
      mv[e] = load_fresh(&tb.movein_n[at * kMoveinPad]);
      rm[e] = load_fresh(&tb.removed_n[at]);
      n[e] = tb.bucket_n[at];
    }
    if (e * (uint32_t)kSlabBlock < P) sn[e] = load_fresh(&tb.serial_n[(x < P ? x : 0u) * kMoveinPad]);
  }
#pragma unroll
  for (uint32_t e = 0; e < kPer; ++e) {
    const uint32_t x = threadIdx.x + e * (uint32_t)kSlabBlock;
    if (x < B) s_start[x] = n[e] + mv[e] - rm[e];
  }
  __syncthreads();
  bool overflow = false;
#pragma unroll
  for (uint32_t e = 0; e < kPer; ++e) {
    const uint32_t x = threadIdx.x + e * (uint32_t)kSlabBlock;
    if (x < P) {
      overflow |= (int64_t)sn[e] > spp;
      s_start[x * geo.bpp + geo.bpp - 1u] += sn[e] > (uint32_t)kSlabSerialCap ? (uint32_t)kSlabSerialCap : sn[e];
    }
  }
  __syncthreads();
  const uint32_t per = (B + (uint32_t)kSlabBlock - 1u) / (uint32_t)kSlabBlock | 1u;  // odd: the lanes on different banks
  const uint32_t first = threadIdx.x * per, end = first + per < B ? first + per : B;
  uint32_t sum = 0;
  for (uint32_t x = first; x < end; ++x) sum += s_start[x];
  uint32_t total;
  uint32_t running = block_exclusive_scan<uint32_t, kSlabBlock>(sum, s_scan, &total);
  for (uint32_t x = first; x < end; ++x) {
    const uint32_t c = s_start[x];
    s_start[x] = running;
    running += c;
  }
  if (threadIdx.x == 0) {
    s_start[B] = total;
    if (total > capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  }
  if (overflow) atomicOr(status, ZEN_STAT_SERIAL_OVERFLOW);
  if (answer.host) wait_global_acks();
  __syncthreads();
  // the split sizes: the host has them while the entries are still on their way to their places
  for (uint32_t p = threadIdx.x; p < P; p += kSlabBlock) {
    const int64_t size = (int64_t)(s_start[(p + 1u) * geo.bpp] - s_start[p * geo.bpp]);
    splits[p] = size;
    if (answer.host) host_store(answer.host + 1 + p, size);
  }
  if (answer.host) {
    if (threadIdx.x == 0)
      host_store(answer.host + 1 + tb.partitions,
                 (int64_t)__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    host_answered(answer);
  }
#pragma unroll
  for (uint32_t e = 0; e < kPer; ++e) {
    const uint32_t x = threadIdx.x + e * (uint32_t)kSlabBlock;
    if (x < B) {
      tb.out_start[x] = s_start[x];
      tb.final_n[x] = mv[e];
      tb.movein_n[x * kMoveinPad] = 0;
    }
    if (x < P) {
      tb.final_n[B + x] = sn[e];
      tb.serial_n[x * kMoveinPad] = 0;
    }
  }
  if (threadIdx.x == 0) tb.out_start[B] = total;
  for (uint32_t x = threadIdx.x; x < kDoneWords; x += kSlabBlock) tb.done[x] = 0;
}

// The way of one index from level `lv` + 1 on, and of those it sets in motion: whoever is pushed out of a slot goes on.
// Those that find no slot are listed in LDS (`serial`, of which one call takes a word at most).
__device__ inline void slab_chain(const SlabGeom &geo, const Probe &g, const SlabTables &tb, unsigned long long *cells,
                                  uint32_t cur, int lv, uint32_t *serial, uint32_t *serial_n, int32_t *status) {
  bool full = false;
  for (uint32_t steps = 0;; ++steps) {
    if (lv >= g.levels) {  // out of levels: cur has no slot
      serial[atomicAdd(serial_n, 1u)] = cur;
      break;
    }
    if (steps > kChainLimit) {
      atomicOr(status, ZEN_STAT_INTERNAL);
      break;
    }
    const SlabGeom::Spot spot = geo.spot(cur, lv);
    const uint32_t bucket = spot.bucket;
    size_t head_pos = 0;
    const uint32_t head = slab_head(geo, tb, spot, &head_pos);
    if (head < cur) {  // a smaller index probes this slot at level 1: cur moves on
      ++lv;
      continue;
    }
    const uint32_t old = part_min(cells, bucket, spot.slot, cur, &full);
    if (full) {
      atomicOr(status, ZEN_STAT_RETRY);
      break;
    }
    if (old < cur) {  // a smaller index got here at level 2 or 3
      ++lv;
      continue;
    }
    if (old == kNone) {
      // first level-2/3 prober of this slot: its level-1 owner (a larger index, if any) is pushed out
      atomicAdd(&tb.movein_n[bucket * kMoveinPad], 1u);
      if (head == kNone) break;
      atomicOr(reinterpret_cast<uint32_t *>(&tb.slab_idx[head_pos]), kRemovedBit);
      atomicAdd(&tb.removed_n[bucket], 1u);
      cur = head;
      lv = 1;
      continue;
    }
    if (old == cur) break;
    // took the slot from a larger index that held it at its first level mapping here
    int lw = 1;
    while (lw < g.levels && geo.spot(old, lw).slot != spot.slot) ++lw;
    cur = old;
    lv = lw + 1;
  }
}

// Level 2 for a group's list of losers.  One in ten or so finds a level-1 owner in its slot: a smaller one sends it on to
// level 3.  The others are entered in the group's parts of the map, which are put together in LDS; whoever finds a smaller
// index there, or is pushed out by one, goes on at level 3 too.  A larger level-1 owner is pushed out by the entry that holds
// its slot in the end, and goes on at level 2.  The owner is asked for first, as a single chain does: a slot with a smaller
// owner takes no cell, and the parts hold no more than the chains alone would put there (16.8 M slots, 27.8 % of them taken,
// 32 partitions: 943 cells in the fullest part; entered first, 1065, more than there are).  Nobody else touches the map
// while this kernel runs.  Bound by latency (four or five trips to memory, as many phases in LDS) and instructions: a group
// to a compute unit, its losers to all of the unit's waves.  62 M slots, 436 000 losers in 256 groups 19.4 us, the chains
// behind it 23.6 (without it the chains 50, and 15 to count the entries that moved in).
template <uint32_t BUCKETS>
struct SlabSettleLds {
  unsigned long long cells[BUCKETS << kSlabPartLog2];
  uint16_t index[BUCKETS * kSlabIndexLen];  // the buckets' indices
  uint32_t in[BUCKETS], pushed[BUCKETS];    // entries that move in, level-1 owners pushed out
  uint32_t tokens;
};

template <int BLOCK, uint32_t BUCKETS>
__global__ __launch_bounds__(BLOCK) void k_slab_settle(SlabGeom geo, SlabTables tb, unsigned long long *cells,
                                                       int32_t *status) {
  static_assert(BUCKETS <= BLOCK, "a thread to a bucket");
  __shared__ SlabSettleLds<BUCKETS> sh;
  constexpr uint32_t mask = (1u << kSlabPartLog2) - 1u;
  const uint32_t group = blockIdx.x, part = group / tb.gpp, first = (group - part * tb.gpp) * tb.per_group;
  const uint32_t b0 = part * geo.bpp + first;
  const uint32_t buckets = geo.bpp - first < tb.per_group ? geo.bpp - first : tb.per_group;
  uint32_t *counter = &tb.group_n[part * tb.group_pad + (group - part * tb.gpp)];
  const uint32_t *list = tb.group_list + (size_t)group * tb.group_cap;
  int32_t *slab_idx = tb.slab_idx + (size_t)b0 * kSlabCap;
  uint32_t *token = tb.token + (size_t)group * tb.group_cap;  // (a loser leaves one at most)
  uint32_t count = *counter;
  const uint16_t *index = tb.sub_index + (size_t)b0 * kSlabIndexLen;
  for (uint32_t i = threadIdx.x; i < buckets * kSlabIndexLen; i += BLOCK) sh.index[i] = index[i];
  count = count < tb.group_cap ? count : tb.group_cap;
  u32x4 *clear = reinterpret_cast<u32x4 *>(sh.cells);
  for (uint32_t i = threadIdx.x; i < (buckets << kSlabPartLog2) / 2u; i += BLOCK) clear[i] = u32x4{0, 0, 0, 0};
  if (threadIdx.x < BUCKETS) sh.in[threadIdx.x] = sh.pushed[threadIdx.x] = 0;
  if (threadIdx.x == 0) sh.tokens = 0;
  __syncthreads();
  if (threadIdx.x == 0) *counter = 0;
  // rows nobody has a loser in are skipped by the whole workgroup; the loads of a step are in flight together
  uint32_t t[kSettleRows];
  SlabGeom::Spot spot[kSettleRows];
  uint32_t in = 0;  // bit r: row r has a loser for this thread that may hold its slot
#pragma unroll
  for (int r = 0; r < kSettleRows; ++r) {
    const uint32_t i = r * BLOCK + threadIdx.x;
    if ((uint32_t)(r * BLOCK) < count) t[r] = list[i < count ? i : 0u];
    in |= (i < count ? 1u : 0u) << r;
  }
  // whose level-1 slot is it: the bucket's index narrows the search to a few records (see slab_head)
  uint32_t head[kSettleRows], pos[kSettleRows], left[kSettleRows], near[kSettleRows][4];
#pragma unroll
  for (int r = 0; r < kSettleRows; ++r) {
    if ((uint32_t)(r * BLOCK) >= count) continue;
    spot[r] = geo.spot(t[r], 1);
    const uint32_t local = spot[r].bucket - b0;
    const uint32_t j = local * kSlabIndexLen + (spot[r].offset >> geo.sub_shift) / (uint32_t)kSlabIndexStep;
    pos[r] = local * (uint32_t)kSlabCap + sh.index[j];
    left[r] = (uint32_t)sh.index[j + 1u] - sh.index[j];
    __builtin_memcpy(near[r], slab_idx + pos[r], sizeof(near[r]));  // (words past the range are not looked at)
  }
  uint32_t cell[kSettleRows];
#pragma unroll
  for (int r = 0; r < kSettleRows; ++r) {
    head[r] = kNone;
    cell[r] = 0;
    if ((uint32_t)(r * BLOCK) >= count || !(in & (1u << r))) continue;
    for (uint32_t at = pos[r];;) {
      bool past = false;
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t v = near[r][q] & kIndexMask;
        const uint32_t s1 = geo.mod_m(poly(v) + kSeed1);
        if (q < left[r] && !past && s1 == spot[r].slot) {
          head[r] = v;
          pos[r] = at + q;
        }
        past |= q < left[r] && s1 >= spot[r].slot;
      }
      if (left[r] <= 4u || past) break;
      left[r] -= 4u;
      at += 4u;
      __builtin_memcpy(near[r], slab_idx + at, sizeof(near[r]));
    }
    if (head[r] < t[r]) {
      in &= ~(1u << r);
      token[atomicAdd(&sh.tokens, 1u)] = t[r] | kAtLevel3;
      continue;
    }
    const uint32_t at = (spot[r].bucket - b0) << kSlabPartLog2;
    const unsigned long long mine = ((unsigned long long)(spot[r].slot + 1u) << 32) | t[r];
    uint32_t h = cell_home(spot[r].slot, kSlabPartLog2), probes = 0;
    for (; probes <= mask; ++probes, h = (h + 1u) & mask) {
      const unsigned long long cur = atomicCAS(&sh.cells[at + h], 0ull, mine);
      if (cur == 0ull) break;
      if (cell_slot(cur) == spot[r].slot) {
        const uint32_t old = (uint32_t)atomicMin(&sh.cells[at + h], mine);
        token[atomicAdd(&sh.tokens, 1u)] = (old < t[r] ? t[r] : old) | kAtLevel3;
        break;
      }
    }
    cell[r] = at + h;
    if (probes > mask) atomicOr(status, ZEN_STAT_RETRY);
  }
  __syncthreads();
  // everybody has entered: who holds the slot moves in, and pushes out a level-1 owner that is there
#pragma unroll
  for (int r = 0; r < kSettleRows; ++r) {
    if ((uint32_t)(r * BLOCK) >= count || !(in & (1u << r)) || (uint32_t)sh.cells[cell[r]] != t[r]) continue;
    const uint32_t local = cell[r] >> kSlabPartLog2;
    atomicAdd(&sh.in[local], 1u);
    if (head[r] != kNone) {
      slab_idx[pos[r]] = (int32_t)(head[r] | kRemovedBit);
      atomicAdd(&sh.pushed[local], 1u);
      token[atomicAdd(&sh.tokens, 1u)] = head[r];
    }
  }
  __syncthreads();
  u32x4 *out = reinterpret_cast<u32x4 *>(cells + ((size_t)b0 << kSlabPartLog2));
  for (uint32_t i = threadIdx.x; i < (buckets << kSlabPartLog2) / 2u; i += BLOCK) {
    const u32x4 q = clear[i];
    if (q.y | q.w) out[i] = q;  // (the map is zero)
  }
  if (threadIdx.x < buckets) {
    tb.movein_n[(b0 + threadIdx.x) * kMoveinPad] = sh.in[threadIdx.x];
    tb.removed_n[b0 + threadIdx.x] = sh.pushed[threadIdx.x];
  }
  if (threadIdx.x == 0) tb.token_n[group] = sh.tokens;
}

// Levels 2 and 3 for the losers on the buckets' lists and for what k_slab_settle has left, one index to a lane, `share`
// workgroups to a group of buckets and as few lanes of a wave as that allows: a wave goes on until the last of them has
// found its place.  Bound by latency: a probe is three or four dependent trips to memory (the bucket's index, its records,
// the map), with a wave to its lanes 1.2 us, and by what all wait for in the end, the layout.  62 M slots, 110 000 losers
// 29.6 -> 26.3 us, 268 M, 18 000 15.8 -> 14.4, 12.9 M, 900 14.9 -> 11.2 (dense waves, a log in one place, divisions, a
// layout by lines of its own to a lane); 72 000 left of 436 000 settled ones 23.6.
__global__ __launch_bounds__(kSlabBlock, 8) void k_slab_chains(SlabGeom geo, Probe g, SlabTables tb, unsigned long long *cells,
                                                            uint32_t share, int64_t spp, uint32_t capacity,
                                                            int64_t *__restrict__ splits, HostAnswer answer,
                                                            int32_t *status) {
  __shared__ uint32_t s_scan[kSlabBlock / 64 + 1];
  __shared__ uint32_t s_start[kSlabMaxBuckets + 1];
  __shared__ uint32_t s_serial, s_first;
  __shared__ bool s_last;
  if (threadIdx.x == 0) s_serial = 0;
  __syncthreads();
  const uint32_t group = blockIdx.x / share, part = group / tb.gpp, first = (group - part * tb.gpp) * tb.per_group;
  const uint32_t b0 = part * geo.bpp + first;
  const uint32_t buckets = geo.bpp - first < tb.per_group ? geo.bpp - first : tb.per_group;
  // lane l of every wave knows where bucket l's list begins among all that there is to do; the tokens come last
  const uint32_t lane = lane_id();
  uint32_t mine = lane < buckets ? tb.again_n[b0 + lane] : 0u;
  if (lane == kGroupBuckets && tb.group_cap) mine = tb.token_n[group];
  const uint32_t incl = wave_inclusive_scan(mine);
  const uint32_t count = (uint32_t)__builtin_amdgcn_readlane((int)incl, kGroupBuckets);
  const uint32_t waves = share * (kSlabBlock / 64), wave = (blockIdx.x - group * share) * (kSlabBlock / 64) + threadIdx.x / 64;
  uint32_t lanes = (count + waves - 1u) / waves;
  lanes = lanes < 64u ? lanes : 64u;
  // (a round has an index to a thread at most: so many are listed at most when the next one begins)
  for (uint32_t i0 = 0; i0 < count; i0 += waves * lanes) {
    const uint32_t i = lane < lanes ? i0 + wave * lanes + lane : count;
    uint32_t list = 0, before = 0;
#pragma unroll
    for (uint32_t l = 0; l < kGroupBuckets; ++l) {
      const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)incl, (int)l);
      if (i >= end) {
        list = l + 1u;
        before = end;
      }
    }
    if (i < count) {
      const uint32_t t = list < kGroupBuckets ? tb.raw_idx[(size_t)(b0 + list) * kSlabCap + (i - before)]
                                              : tb.token[(size_t)group * tb.group_cap + (i - before)];
      slab_chain(geo, g, tb, cells, t & ~kAtLevel3, t & kAtLevel3 ? 2 : 1, s_start, &s_serial, status);
    }
    __syncthreads();
    // those that found no slot, to their partition's list: one atomic (with one each those of a partition stood in line)
    const uint32_t serial = s_serial;
    if (threadIdx.x == 0 && serial) s_first = atomicAdd(&tb.serial_n[part * kMoveinPad], serial);
    __syncthreads();
    if (threadIdx.x < serial) {
      const uint32_t at = s_first + threadIdx.x;
      if (at < (uint32_t)kSlabSerialCap)
        tb.ser_idx[(size_t)part * kSlabSerialCap + at] = s_start[threadIdx.x];
      else  // more than the partition's serial region holds is an overflow; more than this path carries, a retry
        atomicOr(status, (int64_t)at >= spp ? ZEN_STAT_SERIAL_OVERFLOW : ZEN_STAT_RETRY);
    }
    if (threadIdx.x == 0) s_serial = 0;
    __syncthreads();
  }
  // the workgroup that finishes last knows every count and lays out the output
  wait_global_acks();
  __syncthreads();
  if (threadIdx.x == 0) s_last = done_last(tb.done, blockIdx.x, gridDim.x);
  __syncthreads();
  if (s_last) slab_output_starts(geo, tb, s_scan, s_start, spp, capacity, splits, answer, status);
}

// ------------------------------------------------------------------ place

// A bucket's part of the output is its taken slots in order: the owners that nobody pushed out and the entries that moved
// in.  Both are marked in a bitmap of the slots, and an entry goes to the bucket's start plus the number of marks below
// its own.  Consecutive lanes read consecutive entries and write (almost) consecutive places.  62 M slots, 6.2 M records,
// 7 % moved: 34 us (k_slab_place_wide, which counts removed and moved-in entries: 63).
// A partition's overflow entries are a workgroup's own, the first of the launch: sorting them takes longer than placing a
// bucket, and as a part of the partition's last bucket it kept the chip waiting (270 of them on each of 16 partitions, the
// call below: 46 us).
template <uint32_t SPAN>
struct SlabPlaceLds {
  union {
    SlabTaken<SPAN> taken;
    uint32_t serial[kSlabSerialCap];
  };
  uint32_t scan[kSlabBlock / 64 + 1];
};

// The workgroups in front of the buckets': one for every partition, to a multiple of the eight dies, so that a bucket
// stays on the die that sorted it.  Of 1024 partitions few have any: a call of 3 M entries takes 116.5 us with them and 117
// with 256 workgroups of four partitions each; where all have some (one level, 106 000 entries) 112 and 122.
__host__ __device__ inline uint32_t slab_place_lead(uint32_t partitions) { return (partitions + 7u) & ~7u; }

// A partition's overflow entries in ascending index order (the reference hands its tickets to ascending thread ids,
// functions_cuda_kernel.cu:107-108), behind everything that found a slot.
template <typename S>
__device__ inline void slab_place_serial(uint32_t *s_serial, const SlabGeom &geo, const SlabTables &tb, uint32_t part,
                                         const S *__restrict__ dense, int32_t *__restrict__ out_idx,
                                         S *__restrict__ out_val, uint32_t capacity) {
  uint32_t serial = tb.final_n[geo.nbuckets + part];
  if (serial > (uint32_t)kSlabSerialCap) serial = kSlabSerialCap;
  if (serial == 0) return;
  const uint32_t first = tb.out_start[(part + 1u) * geo.bpp] - serial;
  for (uint32_t i = threadIdx.x; i < serial; i += kSlabBlock) s_serial[i] = tb.ser_idx[(size_t)part * kSlabSerialCap + i];
  __syncthreads();
  sort_network(s_serial, serial);
  for (uint32_t i = threadIdx.x; i < serial; i += kSlabBlock) {
    if (first + i < capacity) {
      out_idx[first + i] = (int32_t)s_serial[i];
      out_val[first + i] = dense[s_serial[i]];
    }
  }
}

template <typename S, uint32_t SPAN>
__global__ __launch_bounds__(kSlabBlock, 6) void k_slab_place(SlabGeom geo, SlabTables tb, unsigned long long *cells,
                                                           const S *__restrict__ dense, int32_t *__restrict__ out_idx,
                                                           S *__restrict__ out_val, uint32_t capacity) {
  constexpr int kCells = (1 << kSlabPartLog2) / kSlabBlock;
  __shared__ SlabPlaceLds<SPAN> sh;
  const uint32_t lead = slab_place_lead((uint32_t)tb.partitions);
  if (blockIdx.x < lead) {
    if (blockIdx.x < (uint32_t)tb.partitions)
      slab_place_serial(sh.serial, geo, tb, blockIdx.x, dense, out_idx, out_val, capacity);
    return;
  }
  const uint32_t b = blockIdx.x - lead;
  const size_t base = (size_t)b * kSlabCap;
  const uint32_t words = (geo.span + 63u) / 64u;
  const S *slab_val = static_cast<const S *>(tb.slab_val);
  const uint32_t n = tb.bucket_n[b];
  // what the bucket's part of the map holds has moved in, and keeps to the thread that finds it; the part goes
  // back empty
  const uint32_t mv_n = tb.final_n[b];
  const uint32_t lo = tb.bucket_lo[b];
  const uint32_t out_base = tb.out_start[b];
  unsigned long long *cell = cells + ((size_t)b << kSlabPartLog2) + threadIdx.x;
  unsigned long long moved[kCells];
#pragma unroll
  for (int e = 0; e < kCells; ++e) moved[e] = mv_n ? cell[e * kSlabBlock] : 0ull;
  uint32_t idx[kSlabItems];
  S val[kSlabItems];
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    const uint32_t p = threadIdx.x + i * kSlabBlock;
    idx[i] = kRemovedBit;
    val[i] = 0;
    if ((uint32_t)(i * kSlabBlock) >= n) continue;  // the same for the whole workgroup
    idx[i] = (uint32_t)tb.slab_idx[base + (p < n ? p : 0u)];
    val[i] = slab_val[base + (p < n ? p : 0u)];
    if (p >= n) idx[i] = kRemovedBit;
  }
  sh.taken.template clear<kSlabBlock>(words);
  S mval[kCells];  // an entry is a copy of the element it stands for
#pragma unroll
  for (int e = 0; e < kCells; ++e) mval[e] = mv_n ? dense[(uint32_t)moved[e]] : S(0);
  __syncthreads();
  uint32_t off[kSlabItems], moff[kCells];
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    off[i] = 0;
    if ((uint32_t)(i * kSlabBlock) < n && !(idx[i] & kRemovedBit)) {
      off[i] = geo.mod_m(poly(idx[i]) + kSeed1) - lo;
      sh.taken.take(off[i], 1u);
    }
  }
#pragma unroll
  for (int e = 0; e < kCells; ++e) {
    moff[e] = 0;
    if (moved[e]) {
      cell[e * kSlabBlock] = 0ull;
      moff[e] = cell_slot(moved[e]) - lo;
      sh.taken.take(moff[e], 1u);
    }
  }
  __syncthreads();
  sh.taken.template count<kSlabBlock>(words, sh.scan);  // survivors + moved-in
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    if ((uint32_t)(i * kSlabBlock) < n && !(idx[i] & kRemovedBit)) {
      const uint32_t pos = out_base + sh.taken.place(off[i]);
      if (pos < capacity) {
        out_idx[pos] = (int32_t)idx[i];
        out_val[pos] = val[i];
      }
    }
  }
#pragma unroll
  for (int e = 0; e < kCells; ++e) {
    if (moved[e]) {
      const uint32_t pos = out_base + sh.taken.place(moff[e]);
      if (pos < capacity) {
        out_idx[pos] = (int32_t)(uint32_t)moved[e];
        out_val[pos] = mval[e];
      }
    }
  }
}

// The same for buckets that k_slab_sort_wide has sorted.  A sorted slab is almost the bucket's part of the output
// already: the entries that lost their slot drop out and the entries that moved in from elsewhere slip in between.  So
// an entry at sorted place p goes to
//     bucket start + p - (removed entries before p) + (moved-in entries in front of it).
// A wave's 64 consecutive places are one stretch: how many of its entries in front of a lane's are removed is a
// ballot, how many moved-in ones slip in there a prefix sum across the lanes, and the stretches' sums are chained
// once per bucket.  Consecutive lanes read consecutive entries and write (almost) consecutive places.  (Both counts
// as bisections of sorted lists: 100 us for 6.2 M entries of which 5 % had moved, this 63.)  1.48 G slots, 14.8 M bf16
// records 61 us; 1.34 G and 6.7 M 32.
template <typename S>
__global__ __launch_bounds__(kSlabBlock, 6) void k_slab_place_wide(SlabGeom geo, SlabTables tb,
                                                                unsigned long long *cells,
                                                                const S *__restrict__ dense,
                                                                int32_t *__restrict__ out_idx,
                                                                S *__restrict__ out_val, uint32_t capacity) {
  constexpr int kStretches = kSlabCap / 64;
  constexpr int kCells = (1 << kSlabPartLog2) / kSlabBlock;
  static_assert(kStretches <= 128, "two stretches per lane of a wave");
  __shared__ uint32_t s_key[kSlabCap];                 // sorted slots of the bucket
  __shared__ uint32_t s_cnt[kSlabCap / 2 + 1];         // per sorted place, 16 bits each: the moved-in entries right in
  uint16_t *s_front = reinterpret_cast<uint16_t *>(s_cnt);  // front of it, then those before it in its stretch
  __shared__ uint32_t s_mk[1 << kSlabPartLog2];        // the moved-in entries' slots, by the place they slip in at
  __shared__ uint64_t s_mask[kStretches];              // per stretch: its removed entries
  __shared__ uint32_t s_mv[kStretches], s_rm[kStretches];  // moved-in and removed entries of the stretches before
  __shared__ uint32_t s_nrm;
  const uint32_t b = blockIdx.x;
  const uint32_t B = geo.nbuckets;
  const size_t base = (size_t)b * kSlabCap;
  const S *slab_val = static_cast<const S *>(tb.slab_val);
  const uint32_t *serial_n = tb.final_n + B;
  const uint32_t n = tb.bucket_n[b];
  // what the bucket's part of the map holds has moved in, and keeps to the thread that finds it; the part goes
  // back empty
  const uint32_t mv_n = tb.final_n[b];
  const uint32_t out_base = tb.out_start[b];
  const uint32_t out_n = tb.out_start[b + 1] - out_base;
  unsigned long long *cell = cells + ((size_t)b << kSlabPartLog2) + threadIdx.x;
  unsigned long long moved[kCells];
#pragma unroll
  for (int e = 0; e < kCells; ++e) moved[e] = mv_n ? cell[e * kSlabBlock] : 0ull;
  // the thread's entries (sorted places threadIdx.x + i * kSlabBlock) stay in registers; the slots go to LDS
  // for the searches
  uint32_t idx[kSlabItems];
  S val[kSlabItems];
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    const uint32_t p = threadIdx.x + i * kSlabBlock;
    idx[i] = (uint32_t)tb.slab_idx[base + (p < n ? p : 0u)];
    val[i] = slab_val[base + (p < n ? p : 0u)];
  }
  S mval[kCells];  // an entry is a copy of the element it stands for
#pragma unroll
  for (int e = 0; e < kCells; ++e) mval[e] = mv_n ? dense[(uint32_t)moved[e]] : S(0);
  if (threadIdx.x == 0) s_nrm = 0;
  for (int i = threadIdx.x; i < kSlabCap / 2 + 1; i += kSlabBlock) s_cnt[i] = 0;
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    const uint32_t p = threadIdx.x + i * kSlabBlock;
    if (p < n) s_key[p] = geo.mod_m(poly(idx[i] & kIndexMask) + kSeed1);
  }
  __syncthreads();
  // a moved-in entry's place: the sorted place in front of which it slips in, and its turn among those that slip
  // in there too
  uint32_t mplace[kCells], mturn[kCells];
#pragma unroll
  for (int e = 0; e < kCells; ++e) {
    mplace[e] = mturn[e] = 0;
    if (moved[e]) {
      cell[e * kSlabBlock] = 0ull;
      mplace[e] = lower_bound_u32(s_key, n, cell_slot(moved[e]));
      const uint32_t shift = 16u * (mplace[e] & 1u);
      mturn[e] = (atomicAdd(&s_cnt[mplace[e] >> 1], 1u << shift) >> shift) & 0xffffu;
    }
  }
  __syncthreads();
  uint32_t in_front[kSlabItems];  // moved-in entries of the stretch that slip in at or before the entry's place
  uint32_t removed = 0;           // bit i: entry i has lost its slot
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    const uint32_t p = threadIdx.x + i * kSlabBlock;
    in_front[i] = 0;
    if ((uint32_t)(i * kSlabBlock) > n) {  // the same for the whole workgroup: nothing beyond the entries
      if (lane_id() == 63) s_mv[p >> 6] = s_rm[p >> 6] = 0;
      continue;
    }
    const bool gone = p < n && (idx[i] & kRemovedBit);
    const uint64_t m = __ballot(gone);
    removed |= (gone ? 1u : 0u) << i;
    if (mv_n) {
      const uint32_t c = s_front[p];
      in_front[i] = wave_inclusive_scan(c);
      s_front[p] = (uint16_t)(in_front[i] - c);
    }
    if (lane_id() == 63) {
      s_mask[p >> 6] = m;
      s_mv[p >> 6] = in_front[i];
      s_rm[p >> 6] = (uint32_t)__popcll(m);
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int l = threadIdx.x;
    const uint32_t v0 = s_mv[l], v1 = l + 64 < kStretches ? s_mv[l + 64] : 0u;
    const uint32_t r0 = s_rm[l], r1 = l + 64 < kStretches ? s_rm[l + 64] : 0u;
    const uint32_t iv0 = wave_inclusive_scan(v0), iv1 = wave_inclusive_scan(v1);
    const uint32_t ir0 = wave_inclusive_scan(r0), ir1 = wave_inclusive_scan(r1);
    const uint32_t tv = __shfl(iv0, 63, 64), tr = __shfl(ir0, 63, 64);
    s_mv[l] = iv0 - v0;
    s_rm[l] = ir0 - r0;
    if (l + 64 < kStretches) {
      s_mv[l + 64] = tv + iv1 - v1;
      s_rm[l + 64] = tr + ir1 - r1;
    }
    if (l == 63) s_nrm = tr + ir1;
  }
  __syncthreads();
  // survivors
#pragma unroll
  for (int i = 0; i < kSlabItems; ++i) {
    const uint32_t p = threadIdx.x + i * kSlabBlock;
    if ((uint32_t)(i * kSlabBlock) >= n) break;
    const uint64_t m = __ballot((removed >> i) & 1u);
    if (p < n && !((removed >> i) & 1u)) {
      const uint32_t before = (uint32_t)__popcll(m & lanes_below());
      const uint32_t pos = out_base + p + s_mv[p >> 6] + in_front[i] - s_rm[p >> 6] - before;
      if (pos < capacity) {
        out_idx[pos] = (int32_t)idx[i];
        out_val[pos] = val[i];
      }
    }
  }
  if (mv_n) {  // the same for the whole workgroup
    // the moved-in entries by the place they slip in at; several at one place (two at times) by ascending slot
    const auto front = [&](uint32_t p) -> uint32_t {  // moved-in entries before those of place p
      return p < (uint32_t)kSlabCap ? s_mv[p >> 6] + s_front[p] : p > (uint32_t)kSlabCap ? mv_n : mv_n - s_front[kSlabCap];
    };
#pragma unroll
    for (int e = 0; e < kCells; ++e)
      if (moved[e]) s_mk[front(mplace[e]) + mturn[e]] = cell_slot(moved[e]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kCells; ++e) {
      if (moved[e]) {
        const uint32_t at = mplace[e], key = cell_slot(moved[e]);
        const uint32_t first = front(at), end = front(at + 1u);
        uint32_t rank = first;
        for (uint32_t u = first; u < end; ++u) rank += s_mk[u] < key;
        const uint32_t gone =
            at < n ? s_rm[at >> 6] + (uint32_t)__popcll(s_mask[at >> 6] & ((1ull << (at & 63u)) - 1ull)) : s_nrm;
        const uint32_t pos = out_base + at + rank - gone;
        if (pos < capacity) {
          out_idx[pos] = (int32_t)(uint32_t)moved[e];
          out_val[pos] = mval[e];
        }
      }
    }
  }
  const uint32_t part = b / geo.bpp;
  const bool last_of_part = b % geo.bpp == geo.bpp - 1;
  uint32_t serial = 0;
  if (last_of_part) {
    serial = serial_n[part];
    if (serial > (uint32_t)kSlabSerialCap) serial = kSlabSerialCap;
  }
  const uint32_t own_n = out_n - serial;  // survivors + moved-in
  if (serial) {
    // the partition's overflow entries in ascending index order (the reference hands its tickets to
    // ascending thread ids, functions_cuda_kernel.cu:107-108), behind everything that found a slot
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < serial; i += kSlabBlock) s_key[i] = tb.ser_idx[(size_t)part * kSlabSerialCap + i];
    __syncthreads();
    sort_network(s_key, serial);
    for (uint32_t i = threadIdx.x; i < serial; i += kSlabBlock) {
      const uint32_t pos = out_base + own_n + i;
      if (pos < capacity) {
        out_idx[pos] = (int32_t)s_key[i];
        out_val[pos] = dense[s_key[i]];
      }
    }
  }
}

struct SlabPlan {
  SlabTables tb;
  uint32_t *sample_hist[2];  // sampled floor histogram (+ finished-block count); two sets, so that the sample of
                             // the next call can be taken (zen_load_balance_prepare) while this call still runs
  uint32_t *cand_hist;
  uint32_t *ticket;
  CoarseGeom cg;
  FeedBuffers feed;
  uint32_t *thr;          // [0..1] exact threshold + count, [2..3] sampled floor, [4] candidates above the k-th's bin,
                          // [6..7] sampled floor of the second set
  uint32_t *refine_hist;  // fp32: histogram of the threshold's last 16 bits (+ finished-workgroup count)
  size_t state_bytes;     // of the zero-between-calls memory
  size_t bytes;           // of the workspace
};

// How many of `capacity` entries lose their level-1 slot: a half of capacity^2 / m where slots are drawn evenly, of which the
// hash makes 1.3 to 1.45 times as many where four divides m (1.0 and up at small odd multiples of a large power of two), 0.97
// where it does not, and 0.50 at powers of two, which count in full: settling pays from fewer there.
double slab_losers(uint32_t m, int64_t capacity) {
  const double even = 0.5 * (double)capacity * ((double)capacity / m);
  return (m & 3u) == 0 && (m & (m - 1u)) != 0 ? 1.4 * even : even;
}

bool settled_by_few(int partitions) { return (uint32_t)partitions > kGroupsMost; }

// `state` is memory that is zero between calls (see above); everything else comes out of the workspace.
SlabPlan plan_slab(void *workspace, void *state, const SlabGeom &geo, int partitions, int dtype, int64_t capacity) {
  SlabPlan p;
  const size_t B = geo.nbuckets;
  const int64_t list_cap = list_capacity(capacity);
  const double losers = slab_losers(geo.m, capacity);
  const bool few = settled_by_few(partitions);
  const double from = std::max((few ? kSettleFewFrom : kSettleFrom) * geo.nbuckets, kSettleLeast);
  const bool settled = losers > std::min(from, kSettleAnyway) && geo.span <= kSlabSpan2;
  const uint32_t most = few ? kFewGroupsMost : kGroupsMost;
  uint32_t per = std::min(std::max((geo.nbuckets + kGroupsMost - 1u) / kGroupsMost, kGroupLeast), kGroupBuckets);
  if (settled) {  // (no more groups than the chip takes at a time, where their sizes allow that)
    const uint32_t each = std::max(most / (uint32_t)partitions, 1u);
    per = (geo.bpp + each - 1u) / each;
    per = few ? std::min(per, kFewBuckets) : std::min(std::max(per, kGroupLeast), kGroupBuckets);
  }
  p.tb.per_group = per;
  p.tb.gpp = (geo.bpp + per - 1u) / per;
  p.tb.group_pad = (p.tb.gpp + 31u) & ~31u;
  const size_t groups = (size_t)p.tb.gpp * partitions;
  p.tb.group_cap = 0;
  if (settled) {
    const uint32_t room = (uint32_t)((few ? kFewBlock : kSettleBlock) * kSettleRows);
    p.tb.group_cap = std::min((uint32_t)(1.25 * losers / (double)groups) + 512u, room);
  }
  {
    Carver cv(state);
    p.sample_hist[0] = cv.take<uint32_t>(sampled_floor_zero_bytes() / sizeof(uint32_t));
    p.sample_hist[1] = cv.take<uint32_t>(sampled_floor_zero_bytes() / sizeof(uint32_t));
    p.cand_hist = cv.take<uint32_t>((size_t)kCandHistWords);
    p.ticket = cv.take<uint32_t>(select_stage_ticket_words());
    p.tb.cursor = cv.take<uint32_t>(B);
    p.feed.coarse_cursor = cv.take<uint32_t>(feed_coarse_cursor_words());
    p.tb.movein_n = cv.take<uint32_t>(B * kMoveinPad);
    p.tb.serial_n = cv.take<uint32_t>((size_t)partitions * kMoveinPad);
    p.tb.done = cv.take<uint32_t>(kDoneWords);
    p.tb.group_n = cv.take<uint32_t>(p.tb.group_cap ? (size_t)partitions * p.tb.group_pad : 1);
    p.refine_hist = cv.take<uint32_t>(dtype == ZEN_BF16 ? 1 : (size_t)kRefineWords);
    p.state_bytes = cv.used;
  }
  Carver cv(workspace);
  p.thr = cv.take<uint32_t>(16);
  p.cg = coarse_geometry(geo, list_cap);
  p.feed.coarse_words = cv.take<uint32_t>(feed_coarse_words(p.cg, 2));
  p.tb.bucket_lo = cv.take<uint32_t>(B);
  p.feed.cursor = p.tb.cursor;
  p.feed.bucket_lo = p.tb.bucket_lo;
  p.tb.coarse_cursor = p.feed.coarse_cursor;
  p.tb.refine_hist = nullptr;
  p.tb.partitions = partitions;
  p.tb.out_start = cv.take<uint32_t>(B + 1);
  p.tb.final_n = cv.take<uint32_t>(B + (size_t)partitions);
  p.tb.bucket_n = cv.take<uint32_t>(B);
  p.tb.removed_n = cv.take<uint32_t>(B);
  p.tb.raw_idx = cv.take<uint32_t>(B * kSlabCap);
  p.tb.raw_val = cv.take<char>(B * kSlabCap * (dtype == ZEN_BF16 ? 2 : 4));
  p.tb.slab_idx = cv.take<int32_t>(B * kSlabCap);
  p.tb.slab_val = cv.take<char>(B * kSlabCap * (dtype == ZEN_BF16 ? 2 : 4));
  p.tb.sub_index = cv.take<uint16_t>(B * kSlabIndexLen);
  p.tb.ser_idx = cv.take<uint32_t>((size_t)partitions * kSlabSerialCap);
  p.tb.again_n = cv.take<uint32_t>(B);
  p.tb.group_list = cv.take<uint32_t>(groups * p.tb.group_cap);
  p.tb.token_n = cv.take<uint32_t>(groups);
  p.tb.token = cv.take<uint32_t>(groups * p.tb.group_cap);
  p.bytes = cv.used;
  return p;
}

// SPAN: keys a bucket's bitmap holds; 0: the kernels that compare.
template <typename S, uint32_t SPAN>
int slab_launch_span(const SlabBalanceArgs &a, const SlabGeom &geo, const SlabPlan &p, hipStream_t s) {
  const uint32_t B = geo.nbuckets;
  const uint32_t *filter = a.k > 0 ? p.thr : nullptr;
  const S *dense = static_cast<const S *>(a.input);
  SlabTables tb = p.tb;
  if (a.g.levels < 2) tb.group_cap = 0;  // (nothing to settle)
  {
    ProfScope prof(kProfFeed, s);
    const EncodeSink<S> sink{geo, p.tb.raw_idx, static_cast<S *>(p.tb.raw_val), filter};
    // the select kernel's candidate histogram and ticket counters lie side by side: back to zero here
    const int rc = feed_fine<2, S>(geo, p.cg, sink, p.feed, a.status, s, p.cand_hist,
                                   (uint32_t)(reinterpret_cast<char *>(p.tb.cursor) - reinterpret_cast<char *>(p.cand_hist)) / 4u);
    if (rc != ZEN_OK) return rc;
  }
  {
    ProfScope prof(kProfSlabSort, s);
    if constexpr (SPAN > 0)
      (tb.group_cap ? k_slab_sort<S, SPAN, true> : k_slab_sort<S, SPAN, false>)<<<dim3(B), dim3(kSortBlock), 0, s>>>(geo, tb);
    else
      k_slab_sort_wide<S><<<dim3(B), dim3(kSortBlock), 0, s>>>(geo, tb, a.status);
    ZEN_LAUNCH_CHECK("k_slab_sort");
  }
  {
    ProfScope prof(kProfSlabChains, s);
    const uint32_t groups = tb.gpp * (uint32_t)tb.partitions;
    if (tb.group_cap) {
      if (settled_by_few(tb.partitions))
        k_slab_settle<kFewBlock, kFewBuckets><<<dim3(groups), dim3(kFewBlock), 0, s>>>(geo, tb, a.hash, a.status);
      else
        k_slab_settle<kSettleBlock, kGroupBuckets><<<dim3(groups), dim3(kSettleBlock), 0, s>>>(geo, tb, a.hash, a.status);
      ZEN_LAUNCH_CHECK("k_slab_settle");
    }
    const uint32_t share = std::min(std::max(kChainsResident / groups, 1u), 16u);
    k_slab_chains<<<dim3(groups * share), dim3(kSlabBlock), 0, s>>>(geo, a.g, tb, a.hash, share, a.spp, (uint32_t)a.capacity,
                                                                    a.splits, a.ask.answer, a.status);
    ZEN_LAUNCH_CHECK("k_slab_chains");
    if (a.ask.answer.host) *a.ask.answered = true;
  }
  {
    ProfScope prof(kProfSlabPlace, s);
    if constexpr (SPAN > 0)
      k_slab_place<S, SPAN><<<dim3(slab_place_lead((uint32_t)p.tb.partitions) + B), dim3(kSlabBlock), 0, s>>>(
          geo, p.tb, a.hash, dense, a.out_idx, static_cast<S *>(a.out_val), (uint32_t)a.capacity);
    else
      k_slab_place_wide<S><<<dim3(B), dim3(kSlabBlock), 0, s>>>(geo, p.tb, a.hash, dense, a.out_idx,
                                                                static_cast<S *>(a.out_val), (uint32_t)a.capacity);
    ZEN_LAUNCH_CHECK("k_slab_place");
  }
  return ZEN_OK;
}

template <typename S>
int slab_launch(const SlabBalanceArgs &a, const SlabGeom &geo, const SlabPlan &p, hipStream_t s) {
  if (geo.span <= kSlabSpan1) return slab_launch_span<S, kSlabSpan1>(a, geo, p, s);
  if (geo.span <= kSlabSpan2) return slab_launch_span<S, kSlabSpan2>(a, geo, p, s);
  return slab_launch_span<S, 0>(a, geo, p, s);
}

// The buckets the records call for; where those are too wide for a bitmap, more of them if the records are dense enough
// and that makes them fit.
bool encode_geometry(int64_t m, int partitions, int64_t capacity, SlabGeom *geo) {
  if (!slab_geometry(m, partitions, capacity, kSlabTarget, 0, geo)) return false;
  SlabGeom more;
  // (a few thousand keys below the width: the divisions round the buckets up)
  if (geo->span > kSlabSpan2 && m / kSlabSparse <= capacity &&
      slab_geometry(m, partitions, capacity, kSlabTarget, (int64_t)kSlabSpan2 - 4096, &more) && more.span <= kSlabSpan2)
    *geo = more;
  return true;
}

}  // namespace

size_t slab_balance_bytes(int64_t m, int partitions, int dtype, int64_t capacity) {
  SlabGeom geo;
  if (!encode_geometry(m, partitions, capacity, &geo)) return 0;
  return plan_slab(nullptr, nullptr, geo, partitions, dtype, capacity).bytes;
}

// The hash map takes the first 8 << hash_log2 bytes of the caller's table (at most half of it: zen_load_balance
// sizes the map so), of which every bucket has a part; the counters sit behind it.
size_t slab_state_offset(uint32_t hash_log2) { return align_up((size_t)8 << hash_log2, 256); }

bool slab_balance_fits(int64_t n, int64_t m, int partitions, int dtype, int64_t capacity, int64_t k, SlabGeom *geo) {
  (void)n;
  (void)k;
  if (capacity > 0x1fffffffll) return false;
  SlabGeom g;
  if (!encode_geometry(m, partitions, capacity, &g)) return false;
  // slab_geometry wants m >= 2^22: a table of 16 MB or more, of which the map takes at most half and the
  // counters less than 2 MB
  if (geo) *geo = g;
  return true;
}

// The sample of a coming call, or the clearing of one nobody will pick up.  The sampling memory and the floor
// sit at the head of the zero-between-calls memory and of the workspace whatever the geometry and the path.
int slab_prepare(const SlabBalanceArgs &a, hipStream_t s) {
  char *state = reinterpret_cast<char *>(a.hash) + slab_state_offset(a.hash_log2);
  Carver cs(state);
  uint32_t *sample_hist[2];
  sample_hist[0] = cs.take<uint32_t>(sampled_floor_zero_bytes() / sizeof(uint32_t));
  sample_hist[1] = cs.take<uint32_t>(sampled_floor_zero_bytes() / sizeof(uint32_t));
  Carver cw(a.workspace);
  uint32_t *thr = cw.take<uint32_t>(16);
  const int set = (a.prepared == 2 || a.second) ? 1 : 0;
  uint32_t *floor = thr + 2 + 4 * set;
  if (a.discard) {  // a sample nobody will pick up: its histogram goes back to zero
    launch_fill<uint32_t>(sample_hist[set], 0u, sampled_floor_zero_bytes() / sizeof(uint32_t), s);
    ZEN_LAUNCH_CHECK("slab: discard a sample");
    return ZEN_OK;
  }
  // the sample alone: the floor stays in the workspace until the call proper picks it up
  if (a.k > 0) return topk_sampled_floor(a.input, a.dtype, a.n, a.k, floor, sample_hist[set], s, true);
  return ZEN_OK;
}

int slab_load_balance(const SlabBalanceArgs &a, hipStream_t s) {
  SlabGeom geo;
  if (!slab_balance_fits(a.n, a.g.m, a.partitions, a.dtype, a.capacity, a.k, &geo))
    return fail(ZEN_EINVAL, "slab_load_balance: sizes do not suit the slab layout");
  char *state = reinterpret_cast<char *>(a.hash) + slab_state_offset(a.hash_log2);
  SlabPlan p = plan_slab(a.workspace, state, geo, a.partitions, a.dtype, a.capacity);
  if (slab_state_offset(a.hash_log2) + p.state_bytes > (size_t)a.g.m * sizeof(int32_t))
    return fail(ZEN_EINVAL, "slab_load_balance: table too small for the counters");
  // never with the geometries slab_geometry gives: a bucket spans 16384 slots or more, and there is a cell for about
  // eight slots up to 2^24 cells
  if (((uint64_t)geo.nbuckets << kSlabPartLog2) > (1ull << a.hash_log2)) return fail(ZEN_EINVAL, "slab_load_balance: table too small for the map");
  const bool refine = a.k > 0 && a.dtype == ZEN_F32;
  if (refine) p.tb.refine_hist = p.refine_hist;
  StageArgs sc;
  sc.in = a.input;
  sc.dtype = a.dtype;
  sc.n = a.n;
  sc.thr = a.thr;
  sc.geo = geo;
  sc.cg = p.cg;
  sc.coarse_cursor = p.feed.coarse_cursor;
  sc.coarse_words = p.feed.coarse_words;
  sc.ticket = p.ticket;
  sc.status = a.status;
  int rc;
  const int set = (a.prepared == 2 || a.second) ? 1 : 0;
  uint32_t *floor = p.thr + 2 + 4 * set;
  if (a.only_prepare) return slab_prepare(a, s);
  if (a.k > 0) {
    // one pass: everything at or above a floor estimated from a sample goes to the slabs, the exact
    // threshold is read off the candidates' histogram and applied when the buckets are sorted
    if (a.near_key) {
      // the caller knows about where the threshold lies (an earlier call's): everything from 4/128 of a power
      // of two below that key is a candidate, no sample
      sc.thr = a.near_key;
      sc.floor_margin = a.dtype == ZEN_BF16 ? 4u : 4u << 16;
    } else {
      if (!a.prepared &&
          (rc = topk_sampled_floor(a.input, a.dtype, a.n, a.k, floor, p.sample_hist[set], s, true)) != ZEN_OK)
        return rc;
      sc.thr = floor;
    }
    sc.cand_hist = p.cand_hist;
    sc.pick_k = a.k;
    sc.pick_thr = p.thr;
    sc.pick_above = p.thr + 4;
    sc.thr_copy = refine ? nullptr : a.thr_out;  // fp32: the threshold is not final yet
    sc.clear = p.sample_hist[set];  // the sample kernel is through with its histogram
    sc.clear_words = (uint32_t)(sampled_floor_zero_bytes() / sizeof(uint32_t));
  }
  if (a.next_input && a.next_k > 0) {
    sc.next_in = a.next_input;
    sc.next_k = a.next_k;
    sc.next_n = a.next_n;
    sc.next_hist = p.sample_hist[1 - set];
    if (a.next_state) {  // the sampling memory sits at the head of that table's zero-between-calls memory
      Carver cn(a.next_state);
      uint32_t *first = cn.take<uint32_t>(sampled_floor_zero_bytes() / sizeof(uint32_t));
      uint32_t *second = cn.take<uint32_t>(sampled_floor_zero_bytes() / sizeof(uint32_t));
      sc.next_hist = set ? first : second;
    }
    sc.next_floor = p.thr + 2 + 4 * (1 - set);
  }
  if ((rc = select_stage_slabs(sc, s)) != ZEN_OK) return rc;
  if (refine) {
    const uint32_t refine_parts = p.cg.groups * (uint32_t)kCoarseSplit;
    k_refine_threshold<<<dim3(refine_grid(refine_parts)), dim3(kRefineBlock), 0, s>>>(
        p.cg, 1, p.feed.coarse_cursor, p.feed.coarse_words, static_cast<const uint32_t *>(a.input), p.thr,
        p.thr + 4, (uint32_t)a.k, p.refine_hist, a.thr_out, a.status);
    ZEN_LAUNCH_CHECK("k_refine_threshold");
  }
  if (a.dtype == ZEN_BF16) return slab_launch<uint16_t>(a, geo, p, s);
  return slab_launch<uint32_t>(a, geo, p, s);
}

}  // namespace zen
