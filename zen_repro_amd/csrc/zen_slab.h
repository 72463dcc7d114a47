// Bucket slabs: the layout both fast paths (encode and merge) are built on.
//
// Keys that spread evenly over a range -- level-1 hash slots on the encode
// side, hashed indices arriving at one destination on the merge side -- are
// cut into `nbuckets` contiguous key ranges of equal width.  Every bucket owns
// a slab of kSlabCap records in the workspace.  The producer kernel appends
// records to the slabs in whatever order they turn up (one cursor per bucket,
// reserved once per staged batch and bucket); afterwards one workgroup per
// bucket sorts its slab inside LDS.  Buckets never straddle a partition
// (nbuckets = partitions * buckets-per-partition), so bucket order is output
// order.  A slab that overflows raises ZEN_STAT_RETRY and the caller falls
// back to the general (radix sort) path.
#pragma once

#include <math.h>

#include "zen_common.h"

namespace zen {

constexpr uint32_t kRemovedBit = 1u << 31;  // in a sorted index word: the entry lost its level-1 slot
constexpr uint32_t kIndexMask = kRemovedBit - 1u;

constexpr int kSlabBlock = 512;                       // threads of a per-bucket workgroup (the sort takes twice as many)
constexpr int kSlabItems = 12;                        // records per thread
constexpr int kSlabCap = kSlabBlock * kSlabItems;     // records per slab (6144)
constexpr int kSlabSubs = 4096;                       // narrow key ranges inside a bucket (about one record each)
constexpr int kSlabMaxBlock = 1024;                   // largest workgroup that ranks a slab
constexpr int kSlabGroupLimit = 1024;                 // bounds the rank loop on piled-up keys
constexpr int kSlabMaxBuckets = 4096;
constexpr int kSlabTarget = 3584;                     // records a bucket is sized for (leaves 40 % to spare)
constexpr int kSlabResident = 512;                    // per-bucket workgroups the chip holds at a time (256 CUs x 2)
constexpr int kSlabPartLog2 = 10;                     // entries that may move into one bucket from elsewhere, log2
constexpr int kSlabSerialCap = 4096;                  // overflow entries per partition the fast path carries

struct SlabGeom {
  uint32_t m;         // keys are < m
  uint32_t npp;       // keys per partition (m / partitions)
  uint32_t bpp;       // buckets per partition
  uint32_t bpp_mult;  // floor(bpp * 2^32 / npp)
  uint32_t nbuckets;  // partitions * bpp
  uint32_t span;      // keys of one bucket, at most
  int sub_shift;      // key offset inside a bucket >> sub_shift = narrow range (fewer than kSlabSubs of them)
  float inv_m;        // (1 / m)(1 - 2^-20), rounded down
  float inv_npp;      // the same for npp
  uint32_t npp_mult;  // floor(2^32 / npp)
  double width;       // 2^32 / bpp_mult: keys per bucket, to 53 bits

  // x / d for x < 2^32 and quotients below 2^11, without the long integer division sequence.  `inv` is
  // (1 / d)(1 - 2^-20): the two roundings of the float estimate (each at most 2^-24, relative) cannot lift it
  // above x / d, and it falls short by less than 2^11 * 2^-19: it is the quotient or one less.
  __device__ static inline uint32_t div_small(uint32_t x, uint32_t d, float inv, uint32_t *rem) {
    uint32_t q = (uint32_t)((float)x * inv);
    uint32_t r = x - q * d;
    if (r >= d) {
      r -= d;
      ++q;
    }
    *rem = r;
    return q;
  }
  __device__ inline uint32_t mod_m(uint32_t h) const {  // h % m
    uint32_t r;
    div_small(h, m, inv_m, &r);
    return r;
  }
  __device__ inline uint32_t bucket_of(uint32_t key) const {
    uint32_t local;
    const uint32_t part = div_small(key, npp, inv_npp, &local);
    return part * bpp + __umulhi(local, bpp_mult);
  }
  // ceil(sb * 2^32 / bpp_mult), the first local key of a partition's bucket sb.  The product is within 2^-20 of the
  // true quotient, so rounding it down gives the ceiling or one less.
  __device__ inline uint32_t first_local(uint32_t sb) const {
    const uint32_t lo = (uint32_t)((double)sb * width);
    return lo + (__umulhi(lo, bpp_mult) < sb ? 1u : 0u);
  }
  __device__ inline uint32_t first_key(uint32_t b) const {  // smallest key of bucket b
    const uint32_t part = b / bpp, sb = b - part * bpp;
    return part * npp + first_local(sb);
  }
  // Where index t looks at rehash level 1 or 2: as probe_slot, with the slot's bucket and its offset there, and without a
  // division (x * npp_mult / 2^32 is the quotient or one less).
  struct Spot {
    uint32_t slot, bucket, offset;
  };
  __device__ inline Spot spot(uint32_t t, int level) const {
    const uint32_t h = poly(t);
    uint32_t first;
    const uint32_t part = div_small(mod_m(h + kSeed1), npp, inv_npp, &first);
    const uint32_t x = h + (level == 1 ? kSeed2 : kSeed3);
    uint32_t local = x - __umulhi(x, npp_mult) * npp;
    if (local >= npp) local -= npp;
    const uint32_t sb = __umulhi(local, bpp_mult);
    return Spot{part * npp + local, part * bpp + sb, local - first_local(sb)};
  }
};

inline uint32_t slab_npp_mult(uint32_t npp) { return npp > 1u ? (uint32_t)((1ull << 32) / npp) : 0xffffffffu; }
inline double slab_bucket_width(uint32_t bpp_mult) { return 4294967296.0 / (double)bpp_mult; }

// Host side: geometry for `partitions` partitions of a key space of m keys (m a
// multiple of partitions) expected to hold about `expected` records, its buckets
// good_span keys wide or less where the number of buckets allows that (0: any
// width).  Returns false if the slab layout does not suit these sizes.
inline float slab_inverse_below(uint32_t d) {
  const double want = (1.0 / (double)d) * (1.0 - 1.0 / 1048576.0);
  float f = (float)want;
  while ((double)f > want) f = nextafterf(f, 0.0f);
  return f;
}

inline bool slab_geometry(int64_t m, int partitions, int64_t expected, int target, int64_t good_span, SlabGeom *out) {
  if (m < (1ll << 22) || m > 0x7fffffffll || partitions < 1 || partitions > kSlabMaxBuckets || m % partitions != 0 ||
      expected < 1)
    return false;
  int64_t bpp = ceil_div(expected, (int64_t)target * partitions);
  if (bpp < 1) bpp = 1;
  if (bpp * partitions > kSlabMaxBuckets) bpp = kSlabMaxBuckets / partitions;
  // The per-bucket kernels run in rounds of kSlabResident workgroups, and a workgroup costs much the same whether
  // its slab is half or three quarters full: a bucket count a little above a whole number of rounds wastes most
  // of the last one.  Fewer, fuller buckets then do better, as long as a slab keeps a quarter to spare.
  {
    const int64_t rounds = ceil_div(bpp * partitions, (int64_t)kSlabResident);
    const int64_t fewer = (rounds - 1) * kSlabResident / partitions;
    if (fewer >= 1 && expected / (fewer * partitions) <= (int64_t)kSlabCap * 3 / 4) bpp = fewer;
  }
  const int64_t npp = m / partitions;
  if (good_span > 0) {
    int64_t wanted = ceil_div(npp, good_span);
    if (wanted * partitions > kSlabMaxBuckets) wanted = kSlabMaxBuckets / partitions;
    if (bpp < wanted) bpp = wanted;
  }
  const int64_t nb = bpp * partitions;
  if (expected / nb > (int64_t)kSlabCap * 3 / 4) return false;  // too many records per bucket
  if (npp / bpp < 4 * kSlabSubs) return false;                  // buckets narrower than their sub-ranges
  SlabGeom g;
  g.m = (uint32_t)m;
  g.npp = (uint32_t)npp;
  g.bpp = (uint32_t)bpp;
  g.bpp_mult = (uint32_t)(((uint64_t)bpp << 32) / (uint64_t)npp);
  g.nbuckets = (uint32_t)nb;
  const uint64_t width = ((1ull << 32) + g.bpp_mult - 1) / g.bpp_mult + 1;  // keys per bucket, at most
  g.span = (uint32_t)width;
  g.sub_shift = 0;
  while ((width >> g.sub_shift) >= (uint64_t)kSlabSubs) ++g.sub_shift;
  g.width = slab_bucket_width(g.bpp_mult);
  g.npp_mult = slab_npp_mult(g.npp);
  g.inv_m = slab_inverse_below(g.m);
  g.inv_npp = slab_inverse_below(g.npp);
  *out = g;
  return true;
}

// Shared memory of the in-LDS sort.  slab_rank does not touch `tie`: a caller fills it only after
// slab_rank has returned and has no use for `cnt` from then on, so that the two share their memory:
// LDS decides how many workgroups share a compute unit.
constexpr int kSlabPad = 8;                               // words behind the records that may be read, not looked at
constexpr int kSlabQueueCap = kSlabCap - kSlabSubs - 1;  // large-group records a workgroup sets aside
constexpr int kSlabInline = 4;                            // groups up to this size are ranked by their own threads
constexpr int kSlabPairsFrom = 16;                        // groups up to this size are not counted as pairs
constexpr int kSlabQueueMin = 256;                        // records in larger groups below which nothing is set aside
struct alignas(16) SlabSortShared {
  static constexpr bool kQueue = true;
  static constexpr bool kPairs = false;
  uint32_t key[kSlabCap + kSlabPad];
  union {
    uint32_t tie[kSlabCap + kSlabPad];
    struct {
      uint32_t cnt[kSlabSubs + 1];  // at a multiple of 16 bytes
      uint32_t queue[kSlabQueueCap];  // the rest of the ties' memory: records of large groups (see slab_rank)
    };
  };
  uint32_t scan[kSlabMaxBlock / 64 + 1];
  uint32_t bad;
};
static_assert(kSlabSubs + 1 <= kSlabCap && (kSlabCap + kSlabPad) % 4 == 0, "the counters fit under the ties, and begin at a vector");

// The same without the queue (whose code costs slab_rank registers).
struct alignas(16) SlabSortSharedNoQueue {
  static constexpr bool kQueue = false;
  static constexpr bool kPairs = false;
  uint32_t key[kSlabCap + kSlabPad];
  union {
    uint32_t tie[kSlabCap];
    uint32_t cnt[kSlabSubs + 1];
  };
  uint32_t scan[kSlabMaxBlock / 64 + 1];
  uint32_t bad;
};

// Number of words in words[b0, b1) that are smaller than w.  Four words at a time, all in flight together (a loop that
// fetches one word per turn waits for LDS once per word, and that wait is what such a loop spends its time on); only
// what is left in the end is pulled back onto the last word and checked.  Bound by instructions: 6.2 M bf16 entries of
// sixteen lists, one index in forty in all of them, k_merge_bucket 79 -> 74 us against pulling back and checking all words.
__device__ inline uint32_t count_less(const uint32_t *words, uint32_t b0, uint32_t b1, uint32_t w) {
  uint32_t less = 0, u = b0;
  for (; u + 4u <= b1; u += 4) {
    const uint32_t a0 = words[u], a1 = words[u + 1], a2 = words[u + 2], a3 = words[u + 3];
    less += (a0 < w) + (a1 < w) + (a2 < w) + (a3 < w);
  }
  if (u < b1) {
    const uint32_t last = b1 - 1u;
    const uint32_t a0 = words[u];
    const uint32_t a1 = words[u + 1 < last ? u + 1 : last];
    const uint32_t a2 = words[last];
    less += (a0 < w) + (u + 1 < b1 && a1 < w) + (u + 2 < b1 && a2 < w);
  }
  return less;
}

__device__ inline float value_of(float v) { return v; }
__device__ inline float value_of(uint32_t bits) { return __uint_as_float(bits); }
// The sum, in order from +0, of the sorted records in front of place `first` that share the key k of the one just in front
// of it.  Four records a trip to LDS: 3.1 M bf16 entries of sixteen lists into 62 M elements, k_wide_merge 40.9 -> 39.2 us
// against one.
template <typename V>
__device__ inline float sum_run_before(const uint32_t *key, const V *val, uint32_t first, uint32_t k) {
  uint32_t head = first - 1;
  while (head > 0) {
    const uint32_t a0 = key[head - 1];
    const uint32_t a1 = key[head >= 2 ? head - 2 : 0u];
    const uint32_t a2 = key[head >= 3 ? head - 3 : 0u];
    const uint32_t a3 = key[head >= 4 ? head - 4 : 0u];
    if (a0 != k) break;
    if (head < 2 || a1 != k) { head -= 1; break; }
    if (head < 3 || a2 != k) { head -= 2; break; }
    if (head < 4 || a3 != k) { head -= 3; break; }
    head -= 4;
  }
  float acc = 0.0f;
  uint32_t u = head;
  for (; u + 4u <= first; u += 4) {
    const float f0 = value_of(val[u]), f1 = value_of(val[u + 1]), f2 = value_of(val[u + 2]), f3 = value_of(val[u + 3]);
    acc += f0;
    acc += f1;
    acc += f2;
    acc += f3;
  }
  for (; u < first; ++u) acc += value_of(val[u]);
  return acc;
}

// Ranks the live records of a workgroup of BLOCK threads (ITEMS records each) by (key offset, tie);
// tie < 2^tie_bits, the pair unique, and
// geo.sub_shift + tie_bits <= 32.  off[i] < bucket width.  The records are first grouped by narrow key range
// with one LDS atomic each; a record is then one word, (offset inside the range) << tie_bits | tie, and
// inside its group every record counts the words smaller than its own: the first kSlabInline words of every
// record's group are fetched in one go (all of them in flight together), which settles groups up to that size.
// Where many records share a key (a merge of payloads that overlap) a few lanes of every wave would then walk
// through groups of dozens while the others wait: with a Shared that has a queue, records of groups larger
// than kSlabInline are set aside instead (their places in the queue follow from the same prefix sums as the
// groups' places: the counters carry both, 16 bits each) and handed out again afterwards, one per lane, so
// that the lanes of a wave walk through large groups together.  Returns false (for every thread) if a
// group is too large for that (kSlabGroupLimit; with a Shared that counts pairs: if the records have more than
// sh.pairs_most of others to be compared with, all of them together); else rank[i] for live records and *n_out = number of live records.  On return
// sh.key / sh.tie may be overwritten at once (sh.tie is not touched at all), and the low 16 bits of
// sh.cnt[s] hold the sorted place of the first record of narrow range s.
template <int BLOCK, typename Shared, int ITEMS>
__device__ inline bool slab_rank(Shared &sh, const SlabGeom &geo, int tie_bits,
                                 const uint32_t (&off)[ITEMS], const uint32_t (&tie)[ITEMS],
                                 uint32_t live, uint32_t (&rank)[ITEMS], uint32_t *n_out) {
  static_assert(BLOCK <= kSlabMaxBlock && BLOCK * ITEMS <= kSlabCap, "workgroup size");
  static_assert(kSlabSubs == 4 * BLOCK, "a vector of counters to a thread");
  static_assert(kSlabCap < 65536, "two prefixes in one word");
  uint4 *const cnt4 = reinterpret_cast<uint4 *>(sh.cnt);
  cnt4[threadIdx.x] = make_uint4(0, 0, 0, 0);
  if (threadIdx.x == 0) {
    sh.bad = 0;
    if constexpr (Shared::kPairs) sh.pairs = 0;
  }
  __syncthreads();
  const uint32_t low_mask = (1u << geo.sub_shift) - 1u;
  uint32_t at[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    at[i] = 0;
    if (live & (1u << i)) at[i] = atomicAdd(&sh.cnt[off[i] >> geo.sub_shift], 1u);
  }
  __syncthreads();
  {
    const uint4 q = cnt4[threadIdx.x];
    const uint32_t c[4] = {q.x, q.y, q.z, q.w};
    uint32_t add[4];  // records in the low half, records of groups larger than kSlabInline in the high half
    uint32_t big = 0, pairs = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      add[e] = c[e] | (c[e] > (uint32_t)kSlabInline ? c[e] << 16 : 0u);
      if constexpr (Shared::kPairs)
        pairs += c[e] > (uint32_t)kSlabPairsFrom ? c[e] * c[e] : 0u;
      else
        big |= c[e] > (uint32_t)kSlabGroupLimit;
    }
    if (big) sh.bad = 1;
    if constexpr (Shared::kPairs) {
      if (pairs) atomicAdd(&sh.pairs, pairs);
    }
    uint32_t total;
    const uint32_t b0 = block_exclusive_scan<uint32_t, BLOCK>(add[0] + add[1] + add[2] + add[3], sh.scan, &total);
    const uint32_t b1 = b0 + add[0], b2 = b1 + add[1], b3 = b2 + add[2];
    cnt4[threadIdx.x] = make_uint4(b0, b1, b2, b3);
    if (threadIdx.x == BLOCK - 1) sh.cnt[kSlabSubs] = total;
  }
  __syncthreads();
  if (sh.bad) return false;
  if constexpr (Shared::kPairs) {
    if (sh.pairs > sh.pairs_most) return false;
  }
  const uint32_t totals = (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.cnt[kSlabSubs]);
  // a few large groups are not worth the extra barrier
  const bool set_aside = Shared::kQueue && (totals >> 16) >= (uint32_t)kSlabQueueMin;
  constexpr uint32_t kSetAside = 0x80000000u;
  uint32_t g0[ITEMS], size[ITEMS], word[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    g0[i] = size[i] = word[i] = rank[i] = 0;
    if (live & (1u << i)) {
      const uint32_t sub = off[i] >> geo.sub_shift;
      const uint32_t here = sh.cnt[sub], next = sh.cnt[sub + 1];
      g0[i] = here & 0xffffu;
      size[i] = (next & 0xffffu) - g0[i];
      word[i] = ((off[i] & low_mask) << tie_bits) | tie[i];
      sh.key[g0[i] + at[i]] = word[i];
      if constexpr (Shared::kQueue) {
        static_assert(kSlabSubs <= (1 << 12) && kSlabGroupLimit <= (1 << 19) && kSlabCap <= (1 << 19), "a queue entry is one word");
        if (set_aside) {
          const uint32_t q = (here >> 16) + at[i];
          if (size[i] > (uint32_t)kSlabInline && q < (uint32_t)kSlabQueueCap) {
            sh.queue[q] = sub | (at[i] << 12);  // sub < 2^12, at < group size <= kSlabGroupLimit
            rank[i] = kSetAside | q;
            size[i] = 0;  // nothing left to do for it below
          }
        }
      }
    }
  }
  __syncthreads();
  // the first kAhead words of every record's group (what lies behind the group is read and not looked at), those of kBatch
  // records fetched before any is looked at (most groups are no larger); the rest of a group by count_less
  constexpr int kAhead = Shared::kQueue ? kSlabInline : 2;
  constexpr int kBatch = ITEMS == 4 ? 2 : ITEMS < 3 ? ITEMS : 3;
  static_assert(kAhead <= kSlabPad && kAhead <= 4, "words behind the records");
#pragma unroll
  for (int h = 0; h < ITEMS; h += kBatch) {
    uint32_t a[kBatch][kAhead];
#pragma unroll
    for (int i = 0; i < kBatch && h + i < ITEMS; ++i) {
#pragma unroll
      for (int j = 0; j < kAhead; ++j) a[i][j] = sh.key[g0[h + i] + j];
    }
#pragma unroll
    for (int i = 0; i < kBatch && h + i < ITEMS; ++i) {
      uint32_t less = a[i][0] < word[h + i] ? 1u : 0u;
#pragma unroll
      for (int j = 1; j < kAhead; ++j) less += ((size[h + i] > (uint32_t)j) & (a[i][j] < word[h + i])) ? 1u : 0u;
      if (size[h + i] > (uint32_t)kAhead)
        less += count_less(sh.key, g0[h + i] + kAhead, g0[h + i] + size[h + i], word[h + i]);
      if (!Shared::kQueue || rank[h + i] == 0) rank[h + i] = g0[h + i] + less;
    }
  }
  if constexpr (Shared::kQueue) {
    if (set_aside) {
      const uint32_t queued = (totals >> 16) < (uint32_t)kSlabQueueCap ? (totals >> 16) : (uint32_t)kSlabQueueCap;
      // the thread that takes a queue entry also overwrites it with the rank
#pragma unroll 1
      for (uint32_t q = threadIdx.x; q < queued; q += BLOCK) {
        const uint32_t e = sh.queue[q];
        const uint32_t b0 = sh.cnt[e & 4095u] & 0xffffu;
        const uint32_t b1 = sh.cnt[(e & 4095u) + 1] & 0xffffu;
        sh.queue[q] = b0 + count_less(sh.key, b0, b1, sh.key[b0 + (e >> 12)]);
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < ITEMS; ++i)
        if (rank[i] & kSetAside) rank[i] = sh.queue[rank[i] & ~kSetAside];
    }
  }
  *n_out = totals & 0xffffu;
  __syncthreads();
  return true;
}

// Which keys of a bucket are taken, one bit each, and how many of them lie before every 64th key: a key's place among
// those that are taken is then two look-ups and a count of bits, whatever order the records come in.  SPAN: keys of a
// bucket, at most; `words` of the bitmap's words are in use.
template <uint32_t SPAN>
struct SlabTaken {
  static constexpr uint32_t kWords = (SPAN + 63) / 64;
  uint64_t bits[kWords];
  uint16_t before[kWords];

  template <int BLOCK>
  __device__ inline void clear(uint32_t words) {
    for (uint32_t i = threadIdx.x; i < words; i += BLOCK) bits[i] = 0;
  }
  // Marks key `off`; the bits of its half word before that (`mark` 0: nothing is marked).
  __device__ inline uint32_t take(uint32_t off, uint32_t mark) {
    return atomicOr(reinterpret_cast<uint32_t *>(bits) + (off >> 5), mark << (off & 31u));
  }
  // Fills `before`, by the whole workgroup between barriers; returns the number of keys taken.
  template <int BLOCK>
  __device__ inline uint32_t count(uint32_t words, uint32_t *scan) {
    const uint32_t per = (words + BLOCK - 1) / BLOCK | 1u;  // odd: the lanes of a wave on different banks
    const uint32_t first = threadIdx.x * per, end = first + per < words ? first + per : words;
    uint32_t sum = 0;
    for (uint32_t i = first; i < end; ++i) sum += (uint32_t)__popcll(bits[i]);
    uint32_t total;
    uint32_t run = block_exclusive_scan<uint32_t, BLOCK>(sum, scan, &total);
    for (uint32_t i = first; i < end; ++i) {
      before[i] = (uint16_t)run;
      run += (uint32_t)__popcll(bits[i]);
    }
    return total;
  }
  // Keys taken below `off`.
  __device__ inline uint32_t place(uint32_t off) const {
    return before[off >> 6] + (uint32_t)__popcll(bits[off >> 6] & ((1ull << (off & 63u)) - 1ull));
  }
};

}  // namespace zen
