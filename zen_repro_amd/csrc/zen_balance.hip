// Hash partitioning: hash_index, the in-place table insert (sparse_balance) and
// the fused select + insert + slot-order compaction (load_balance).
//
// The reference insert (functions_cuda_kernel.cu:97-167) is a race: plain load,
// plain store.  Run with its threads in ascending order it has one well-defined
// result: a slot belongs to the smallest index that ever probes it, and an
// index probes level l+1 only if a smaller index owns its level-l slot.  That
// fixed point is computed here by letting the smallest index win every slot: a
// thread that takes a slot from a larger index carries on with that index's probe
// sequence, so every lost probe is continued exactly once and no rounds or flags
// are needed.  In the library's own tables the winner is found with atomicMax on
// the encoding 0 - index (so the empty marker 0 stays the smallest value).
#include "zen_balance.h"
#include "zen_hashmap.h"
#include "zen_wide.h"

namespace zen {
namespace {

__device__ inline void insert_chain(uint32_t *table, const Probe &g, uint32_t t) {
  uint32_t cur = t;
  int lv = 0;
  for (;;) {
    uint32_t part;
    const uint32_t slot = probe_slot(g, cur, lv, &part);
    const uint32_t mine = 0u - cur;
    const uint32_t old = atomicMax(&table[slot], mine);
    if (old > mine) {  // a smaller index owns the slot: cur moves on
      if (++lv >= g.levels) return;  // out of levels: found later by its absence
      continue;
    }
    if (old == 0u || old == mine) return;  // took an empty slot
    // took the slot from a larger index w: w held it at its first level that
    // maps here, and now continues from the next one
    const uint32_t w = 0u - old;
    int lw = 0;
    while (lw < g.levels && probe_slot(g, w, lw, &part) != slot) ++lw;
    cur = w;
    lv = lw + 1;
    if (lv >= g.levels) return;
  }
}

// level at which t holds a slot, or -1; *slot_out / *part_out as found
__device__ inline int find_level(const uint32_t *table, const Probe &g, uint32_t t, uint32_t *slot_out,
                                 uint32_t *part_out) {
  const uint32_t mine = 0u - t;
  for (int lv = 0; lv < g.levels; ++lv) {
    const uint32_t slot = probe_slot(g, t, lv, part_out);
    if (table[slot] == mine) {
      *slot_out = slot;
      return lv;
    }
  }
  return -1;
}

// ------------------------------------------------------------- hash_index

__global__ __launch_bounds__(256) void k_hash_index(int32_t *__restrict__ out, uint32_t n, uint32_t per_part) {
  for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < n; t += gridDim.x * 256u)
    out[t] = (int32_t)(((poly(t) + kSeed1) % n) / per_part);
}

// ------------------------------------------------ in-place insert (dense)

// The same chain in a table of plain indices, as the caller gets it: an empty slot is claimed with a compare-and-swap, an
// occupied one never becomes empty again, so that from then on the minimum decides.  Returns the index that ends up
// without a slot (0: none) and its partition.
__device__ inline uint32_t insert_plain(uint32_t *table, const Probe &g, uint32_t t, uint32_t *part) {
  uint32_t cur = t;
  int lv = 0;
  for (;;) {
    const uint32_t slot = probe_slot(g, cur, lv, part);
    uint32_t old = atomicCAS(&table[slot], 0u, cur);
    if (old > cur) old = atomicMin(&table[slot], cur);
    if (old == 0u || old == cur) return 0;
    if (old < cur) {  // a smaller index owns the slot: cur moves on
      if (++lv >= g.levels) return cur;
      continue;
    }
    // took the slot from a larger index, which goes on behind its first level that maps here
    cur = old;
    lv = 0;
    while (lv < g.levels && probe_slot(g, cur, lv, part) != slot) ++lv;
    if (++lv >= g.levels) return cur;
  }
}

// Bound by the atomics, one or a few per index at random places: 21 a nanosecond.  (On 0 - index with a maximum, which
// needed a second kernel that looked every index up again, wrote it as it is and found those without a slot: 16.8 M
// bf16 elements, 5 % nonzero: 39 + 33 us.)  The indices without a slot are collected per workgroup, and a wave asks for
// the places of all partitions at once: the partitions' counters lie side by side, and one line carries out a request
// every ten nanoseconds (a request per index, 2.3 M bf16 elements on 8 partitions, 10 % nonzero, one level: 151 us).
constexpr int kDenseBlock = 512;
constexpr uint32_t kDenseLost = 2048;   // indices without a slot a workgroup collects; the others ask one by one
constexpr int kDenseParts = 1024;       // partitions up to which it collects

template <typename S, bool ALIGNED>
__global__ __launch_bounds__(kDenseBlock) void k_insert_dense(const S *__restrict__ in, int64_t n, uint32_t *table, Probe g,
                                                              int32_t *serial, int64_t spp, int32_t *offset, int partitions,
                                                              int32_t *status) {
  constexpr int V = VecOf<S>::kN;
  __shared__ uint32_t lost_t[kDenseLost], lost_at[kDenseLost];  // the index; partition << 16 | place among its partition's
  __shared__ int32_t held[kDenseParts];                         // collected per partition, then where they go
  __shared__ uint32_t lost_n;
  static_assert(kDenseLost <= 65536, "a place in 16 bits");
  const bool collect = partitions <= kDenseParts;
  if (collect)
    for (int p = threadIdx.x; p < partitions; p += kDenseBlock) held[p] = 0;
  if (threadIdx.x == 0) lost_n = 0;
  __syncthreads();
  auto put = [&](uint32_t t, uint32_t part, int64_t ticket) {
    if (ticket >= 0 && ticket < (int64_t)(part + 1) * spp)
      serial[ticket] = (int32_t)t;
    else
      atomicOr(status, ZEN_STAT_SERIAL_OVERFLOW);
  };
  const int64_t nvec = (n + V - 1) / V;
  for (int64_t v = blockIdx.x * (int64_t)kDenseBlock + threadIdx.x; v < nvec; v += (int64_t)gridDim.x * kDenseBlock) {
    S e[V];
    const int live = load_vec<S, ALIGNED>(in, v * V, n, e);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const uint32_t t = (uint32_t)(v * V + i);
      if (!(i < live && (e[i] & KeyOf<S>::kMask) != 0 && t != 0)) continue;
      uint32_t part;
      const uint32_t left = insert_plain(table, g, t, &part);
      if (left == 0) continue;
      const uint32_t at = collect ? atomicAdd(&lost_n, 1u) : kDenseLost;
      if (at < kDenseLost) {
        lost_t[at] = left;
        lost_at[at] = (part << 16) | (uint32_t)atomicAdd(&held[part], 1);
      } else {
        put(left, part, atomicAdd(&offset[part], 1));
      }
    }
  }
  __syncthreads();
  const uint32_t lost = lost_n < kDenseLost ? lost_n : kDenseLost;
  if (!collect || lost == 0) return;
  for (int p = threadIdx.x; p < partitions; p += kDenseBlock)
    if (held[p]) held[p] = atomicAdd(&offset[p], held[p]);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < lost; i += kDenseBlock) {
    const uint32_t part = lost_at[i] >> 16;
    put(lost_t[i], part, (int64_t)held[part] + (lost_at[i] & 0xffffu));
  }
}

// Tickets are handed out in arrival order; the canonical order is ascending
// index inside each partition's region, so each region is sorted in place.
//
// A region's indices lie anywhere in [0, n), spread as evenly as the nonzeros are: they are grouped by narrow index
// ranges in LDS (WideCounters, zen_wide.h) and ranked against the few words of their range, a part of them at a time
// and the rest in the workgroup's registers.  Bound by the LDS round trips, a dozen for every 16 384 entries: 4
// regions of 5200 entries 12 us, 4 of 21 000 17 (the compare-exchange network: 68 and, in memory, several hundred).  Where the indices pile up, and
// for more than 64 512, the network does it.
constexpr int kSerialSortBlock = 1024;
constexpr uint32_t kRangeSort = 8192;       // entries expected in one go where there are more than there is room for (16 384):
                                            // the larger of two indices loses, so that the last range holds up to twice its share
constexpr uint32_t kRangeGroup = 64;        // entries of a narrow range, at most
struct SerialSortShared {
  WideCounters cnt;
  uint32_t key[kWideSubs];
  uint32_t scan[kSerialSortBlock / 64 + 1];
  uint32_t big;
};

// Whether the region's cnt <= ITEMS * kSerialSortBlock entries could be put in order (else they are as they were).
template <int ITEMS>
__device__ inline bool sort_spread(uint32_t *region, uint32_t cnt, uint32_t n, SerialSortShared &sh) {
  const uint32_t tid = threadIdx.x;
  uint32_t k[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t j = tid + (uint32_t)(i * kSerialSortBlock);
    k[i] = kNone;
    if ((uint32_t)(i * kSerialSortBlock) < cnt) k[i] = j < cnt ? region[j] : kNone;
  }
  const uint32_t turns = cnt <= (uint32_t)kWideSubs ? 1u : (cnt + kRangeSort - 1u) / kRangeSort, width = (n - 1u) / turns + 1u;
  uint32_t shift = 0, placed = 0;
  while (((width - 1u) >> shift) >= (uint32_t)kWideSubs) ++shift;
  bool ok = true;
  for (uint32_t r = 0; r < turns; ++r) {
    const uint32_t lo = r * width;  // (an entry's distance from it wraps around below)
    sh.cnt.clear();
    if (tid == 0) sh.big = 0;
    __syncthreads();  // (and everybody holds the entries of the last turn in registers)
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
      if ((uint32_t)(i * kSerialSortBlock) < cnt && k[i] != kNone && k[i] - lo < width) sh.cnt.count((k[i] - lo) >> shift);
    __syncthreads();
    const uint32_t here = sh.cnt.starts(sh.scan, kRangeGroup, &sh.big);
    __syncthreads();
    if (here > (uint32_t)kWideSubs || sh.big) {
      ok = false;
      break;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
      if ((uint32_t)(i * kSerialSortBlock) < cnt && k[i] != kNone && k[i] - lo < width) sh.key[sh.cnt.take((k[i] - lo) >> shift)] = k[i];
    __syncthreads();
    for (uint32_t j = tid; j < here; j += kSerialSortBlock) {
      const uint32_t mine = sh.key[j], sub = (mine - lo) >> shift, end = sh.cnt.end_of(sub);
      uint32_t at = sh.cnt.start_of(sub);
      for (uint32_t u = at; u < end; ++u) at += sh.key[u] < mine;
      region[placed + at] = mine;
    }
    placed += here;
    __syncthreads();
  }
  if (ok) return true;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    if (k[i] != kNone) region[tid + (uint32_t)(i * kSerialSortBlock)] = k[i];
  __syncthreads();
  return false;
}

__global__ __launch_bounds__(kSerialSortBlock) void k_serial_sort(int32_t *serial, int64_t spp, const int32_t *offset,
                                                                  uint32_t n) {
  __shared__ SerialSortShared sh;
  const int p = blockIdx.x;
  const int64_t begin = (int64_t)p * spp;
  int64_t end = offset[p];
  if (end > begin + spp) end = begin + spp;
  if (end - begin < 2) return;
  const uint32_t cnt = (uint32_t)(end - begin);
  uint32_t *region = reinterpret_cast<uint32_t *>(serial + begin);
  if (cnt <= 16u * kSerialSortBlock) {
    if (sort_spread<16>(region, cnt, n, sh)) return;
    for (uint32_t i = threadIdx.x; i < cnt; i += kSerialSortBlock) sh.key[i] = region[i];
    __syncthreads();
    sort_network(sh.key, cnt);
    for (uint32_t i = threadIdx.x; i < cnt; i += kSerialSortBlock) region[i] = sh.key[i];
  } else if (cnt > 63u * kSerialSortBlock || !sort_spread<63>(region, cnt, n, sh)) {  // (counts below 2^16)
    sort_network(region, cnt);
  }
}

// ------------------------------------------------- fused path (list based)

template <typename S>
__global__ __launch_bounds__(256) void k_insert_list(const int32_t *__restrict__ cand, const S *__restrict__ vals,
                                                     const uint32_t *count, const uint32_t *__restrict__ thr,
                                                     uint32_t *table, Probe g) {
  const uint32_t j = blockIdx.x * 256u + threadIdx.x;
  if (j >= *count) return;
  uint32_t t;
  if (list_selected<S>(cand, vals, thr, j, &t)) insert_chain(table, g, t);
}

// Sort key = position in the output: partition-major, table slots before the
// partition's serial entries (all serial entries of a partition share one key).
template <typename S>
__global__ __launch_bounds__(256) void k_final_key(const int32_t *__restrict__ cand, const S *__restrict__ vals,
                                                   const uint32_t *count, const uint32_t *__restrict__ thr,
                                                   const uint32_t *__restrict__ table, Probe g, uint32_t drop_key,
                                                   uint32_t *__restrict__ keys, uint32_t *__restrict__ perm) {
  const uint32_t j = blockIdx.x * 256u + threadIdx.x;
  if (j >= *count) return;
  uint32_t t;
  uint32_t key = drop_key;
  if (list_selected<S>(cand, vals, thr, j, &t)) {
    uint32_t slot = 0, part = 0;
    const int lv = find_level(table, g, t, &slot, &part);
    key = part * (g.npp + 1u) + (lv >= 0 ? slot - part * g.npp : g.npp);
  }
  keys[j] = key;
  perm[j] = j;
}

template <typename S>
__global__ __launch_bounds__(256) void k_gather(const uint32_t *__restrict__ keys, const uint32_t *__restrict__ perm,
                                                const uint32_t *count, const int32_t *__restrict__ cand_idx,
                                                const S *__restrict__ cand_val, uint32_t drop_key, Probe g,
                                                int32_t *__restrict__ out_idx, S *__restrict__ out_val,
                                                uint32_t capacity, uint32_t *table) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= *count) return;
  const uint32_t key = keys[i];
  if (key >= drop_key) return;
  const uint32_t j = perm[i];
  if (i < capacity) {
    out_idx[i] = cand_idx[j];
    out_val[i] = cand_val[j];
  }
  const uint32_t part = key / (g.npp + 1u), local = key % (g.npp + 1u);
  if (local < g.npp) table[part * g.npp + local] = 0u;  // leave the table empty again
}

// One block per partition: its length from the sorted keys, and the canonical
// order of its serial tail.  The selected list arrives tile by tile in no
// particular order and all serial entries of a partition share one sort key, so
// the stable sort leaves them in arrival order; the reference order (tickets
// handed out to ascending indices) is restored by sorting the tail by index and
// fetching the values again.
template <typename S>
__global__ __launch_bounds__(256) void k_splits_serial(const uint32_t *__restrict__ keys, const uint32_t *count,
                                                       uint32_t npp, int64_t spp, uint32_t capacity,
                                                       const S *__restrict__ dense, int32_t *__restrict__ out_idx,
                                                       S *__restrict__ out_val, int64_t *__restrict__ splits,
                                                       int32_t *status) {
  __shared__ uint32_t s_bound[3];
  __shared__ uint32_t buf[kSerialLds];
  const uint32_t p = blockIdx.x;
  if (threadIdx.x < 3) {
    const uint32_t first = p * (npp + 1u);
    const uint32_t probe = threadIdx.x == 0 ? first : (threadIdx.x == 1 ? first + npp : first + npp + 1u);
    s_bound[threadIdx.x] = lower_bound_u32(keys, *count, probe);
  }
  __syncthreads();
  const uint32_t lo = s_bound[0], ser = s_bound[1], hi = s_bound[2];
  if (threadIdx.x == 0) {
    splits[p] = (int64_t)(hi - lo);
    if ((int64_t)(hi - ser) > spp) atomicOr(status, ZEN_STAT_SERIAL_OVERFLOW);
    if (hi > capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  }
  if (hi > capacity) return;
  fix_serial_tail<S>(out_idx, out_val, dense, ser, hi - ser, buf);
}

// Fresh tables for an insert: zeros, and where every partition's serial region starts.  One launch in the place of four
// (a fill each, a range and a product), bound by the write: 16.8 M slots 12 us, as the fill alone.
__global__ __launch_bounds__(256) void k_new_tables(uint32_t *__restrict__ table, int64_t m, uint32_t *__restrict__ serial,
                                                    int64_t serial_n, int32_t *__restrict__ offset, int partitions, int64_t spp) {
  const int64_t first = blockIdx.x * (int64_t)256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  auto clear = [&](uint32_t *p, int64_t n) {
    const int64_t head = (int64_t)((16u - (reinterpret_cast<uintptr_t>(p) & 15u)) & 15u) / 4;
    const int64_t skip = head < n ? head : n, vecs = (n - skip) / 4;
    uint4 *v = reinterpret_cast<uint4 *>(p + skip);
    for (int64_t i = first; i < vecs; i += step) v[i] = make_uint4(0, 0, 0, 0);
    if (first < skip) p[first] = 0;
    if (first < n - skip - vecs * 4) p[skip + vecs * 4 + first] = 0;
  };
  clear(table, m);
  clear(serial, serial_n);
  for (int64_t p = first; p < partitions; p += step) offset[p] = (int32_t)(p * spp);
}

template <typename S>
int sparse_balance_launch(const S *in, int64_t n, uint32_t *table, Probe g, int32_t *serial, int64_t spp,
                          int32_t *offset, int partitions, int32_t *status, hipStream_t s) {
  constexpr int V = VecOf<S>::kN;
  const int64_t nvec = ceil_div(n, V);
  int64_t blocks = ceil_div(nvec, kDenseBlock);
  if (blocks > 1024) blocks = 1024;  // as many as the chip holds
  const bool aligned = (reinterpret_cast<uintptr_t>(in) & 15u) == 0;
  ProfScope prof(kProfInsertDense, s);
  if (aligned)
    k_insert_dense<S, true><<<dim3((unsigned)blocks), dim3(kDenseBlock), 0, s>>>(in, n, table, g, serial, spp, offset, partitions, status);
  else
    k_insert_dense<S, false><<<dim3((unsigned)blocks), dim3(kDenseBlock), 0, s>>>(in, n, table, g, serial, spp, offset, partitions, status);
  ZEN_LAUNCH_CHECK("k_insert_dense");
  if (spp > 0) {
    k_serial_sort<<<dim3((unsigned)partitions), dim3(kSerialSortBlock), 0, s>>>(serial, spp, offset, (uint32_t)n);
    ZEN_LAUNCH_CHECK("k_serial_sort");
  }
  return ZEN_OK;
}

constexpr int64_t kSampleMinElems = 1ll << 24;  // below this the exact full-tensor histogram is cheap anyway

struct BalancePlan {
  int32_t *sel_idx;    // the selected entries or candidates (list_capacity)
  uint32_t *sel_val;   // 4 bytes per value reserved, bf16 uses half
  uint32_t *keys_a, *perm_a, *more_a, *keys_b, *perm_b, *more_b;
  uint32_t *count;     // entries in sel_*
  uint32_t *thr;       // [0..1] exact threshold + count, [2..3] sampled floor
  uint32_t *cand_hist;
  void *topk_scratch;
  void *select_scratch;
  void *sort_scratch;
  void *resolve_scratch;
  size_t bytes;
};

BalancePlan plan_balance(void *workspace, int64_t n, int64_t m, int dtype, int64_t capacity) {
  Carver cv(workspace);
  BalancePlan p;
  const size_t cap = (size_t)list_capacity(capacity > 0 ? capacity : 1);
  p.sel_idx = cv.take<int32_t>(cap);
  p.sel_val = cv.take<uint32_t>(cap);
  p.keys_a = cv.take<uint32_t>(cap);
  p.perm_a = cv.take<uint32_t>(cap);
  p.keys_b = cv.take<uint32_t>(cap);
  p.perm_b = cv.take<uint32_t>(cap);
  p.more_a = cv.take<uint32_t>(cap);
  p.more_b = cv.take<uint32_t>(cap);
  p.count = cv.take<uint32_t>(2);
  p.thr = cv.take<uint32_t>(4);
  p.cand_hist = cv.take<uint32_t>((size_t)kCandHistWords);
  p.topk_scratch = cv.take<char>(topk_scratch_bytes());
  p.select_scratch = cv.take<char>(select_scratch_bytes());
  p.sort_scratch = cv.take<char>(sort_scratch_bytes((int64_t)cap));
  // m + P + 1 <= 2 m + 1 bounds the final-position keys whatever the partition count
  p.resolve_scratch = cv.take<char>(resolve_scratch_bytes((int64_t)cap, 2ull * (uint64_t)m + 1));
  p.bytes = cv.used;
  return p;
}

// Stage 1 of load balance: an (index, value) list in p.sel_* with its length in
// p.count[0], and in *filter the threshold the later stages must still apply to
// it (nullptr: every entry is selected).  k > 0 asks for the k largest
// magnitudes (ties at the threshold kept); the threshold goes to p.thr[0..1].
int select_stage(const BalancePlan &p, const void *input, int dtype, int64_t n, const uint32_t *thr, int64_t k,
                 int64_t capacity, int mode, const uint32_t **filter, int32_t *status, hipStream_t s) {
  SelectArgs sel;
  sel.in = input;
  sel.dtype = dtype;
  sel.n = n;
  sel.thr = thr;
  sel.out_idx = p.sel_idx;
  sel.out_val = p.sel_val;
  sel.capacity = list_capacity(capacity);
  sel.out_count32 = &p.count[0];
  sel.scratch = p.select_scratch;
  sel.status = status;
  *filter = nullptr;
  if (k <= 0) return select_compact(sel, s);
  int rc;
  if (mode == ZEN_MODE_GENERAL || n < kSampleMinElems) {
    // exact radix select over the whole tensor, then one compaction pass
    if ((rc = topk_exact(input, dtype, n, nullptr, k, p.thr, p.topk_scratch, status, 0, s)) != ZEN_OK) return rc;
    sel.thr = p.thr;
    return select_compact(sel, s);
  }
  // one pass: compact everything at or above a floor estimated from a sample,
  // histogram those candidates on the way, read the exact threshold off the
  // histogram; entries between floor and threshold stay in the list and are
  // filtered by the later stages
  if ((rc = topk_sampled_floor(input, dtype, n, k, p.thr + 2, p.topk_scratch, s)) != ZEN_OK) return rc;
  launch_fill<uint32_t>(p.cand_hist, 0u, (size_t)kCandHistWords, s);
  ZEN_LAUNCH_CHECK("clear candidate histogram");
  sel.thr = p.thr + 2;
  sel.cand_hist = p.cand_hist;
  sel.pick_k = k;
  sel.pick_thr = p.thr;
  if ((rc = select_compact(sel, s)) != ZEN_OK) return rc;
  if (dtype == ZEN_F32) {
    // the histogram resolved 15 key bits; the remaining 16 need the radix select, over the candidates only
    if ((rc = topk_exact(p.sel_val, dtype, sel.capacity, &p.count[0], k, p.thr, p.topk_scratch, status,
                         ZEN_STAT_RETRY, s)) != ZEN_OK)
      return rc;
  }
  *filter = p.thr;
  return ZEN_OK;
}

}  // namespace
}  // namespace zen

extern "C" {

int zen_hash_index(int32_t *out, int64_t n, int partitions, void *stream) {
  using namespace zen;
  if (!out) return fail(ZEN_EINVAL, "zen_hash_index: null pointer");
  if (n <= 0 || n > 0x7fffffffll || partitions <= 0 || n / partitions == 0)
    return fail(ZEN_EINVAL, "zen_hash_index: need 0 < partitions <= n < 2^31");
  int64_t blocks = ceil_div(n, 256 * 4);
  if (blocks > 65536) blocks = 65536;
  k_hash_index<<<dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
      out, (uint32_t)n, (uint32_t)(n / partitions));
  ZEN_LAUNCH_CHECK("k_hash_index");
  return ZEN_OK;
}

int zen_sparse_balance(const void *input, int dtype, int64_t n, int32_t *memory, int64_t m, int32_t *serial,
                       int64_t serial_n, int32_t *offset, int partitions, int rehash, int32_t *status,
                       void *stream) {
  using namespace zen;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_sparse_balance: bad dtype");
  if (n < 0 || n > 0x7fffffffll || m <= 0 || m > 0x7fffffffll || partitions <= 0 || m % partitions != 0 ||
      serial_n < 0 || serial_n > 0x7fffffffll)
    return fail(ZEN_EINVAL, "zen_sparse_balance: need n, m < 2^31 and m a positive multiple of partitions");
  if (n == 0) return ZEN_OK;
  if (!input || !memory || !offset || !status || (serial_n > 0 && !serial))
    return fail(ZEN_EINVAL, "zen_sparse_balance: null pointer");
  Probe g;
  g.m = (uint32_t)m;
  g.npp = (uint32_t)(m / partitions);
  g.levels = (rehash == 2 || rehash == 3) ? rehash : 1;  // functions_cuda_kernel.cu:192-198
  const int64_t spp = serial_n / partitions;
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint32_t *table = reinterpret_cast<uint32_t *>(memory);
  if (dtype == ZEN_BF16)
    return sparse_balance_launch(static_cast<const uint16_t *>(input), n, table, g, serial, spp, offset,
                                 partitions, status, s);
  return sparse_balance_launch(static_cast<const uint32_t *>(input), n, table, g, serial, spp, offset,
                               partitions, status, s);
}

int zen_balance_tables(const void *input, int dtype, int64_t n, int32_t *memory, int64_t m, int32_t *serial,
                       int64_t serial_n, int32_t *offset, int partitions, int rehash, int32_t *status, int64_t *host,
                       int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  int rc = host_ask(host, words, 1, &answer);
  if (rc != ZEN_OK) return rc;
  if (n < 0 || m <= 0 || m > 0x7fffffffll || partitions <= 0 || serial_n < 0 || serial_n > 0x7fffffffll)
    return fail(ZEN_EINVAL, "zen_balance_tables: need n, m < 2^31 and m a positive multiple of partitions");
  if (!memory || !offset || !status || (serial_n > 0 && !serial)) return fail(ZEN_EINVAL, "zen_balance_tables: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t blocks = ceil_div(m, (int64_t)256 * 4);
  k_new_tables<<<dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(256), 0, s>>>(
      reinterpret_cast<uint32_t *>(memory), m, reinterpret_cast<uint32_t *>(serial), serial_n, offset, partitions,
      serial_n / partitions);
  const hipError_t e = hipGetLastError();
  rc = e == hipSuccess ? zen_sparse_balance(input, dtype, n, memory, m, serial, serial_n, offset, partitions, rehash, status, stream)
                       : hip_fail(e, "k_new_tables");
  if (rc == ZEN_OK) rc = host_answer_launch(answer, nullptr, 0, status, 1, s);
  return host_finish(rc, answer, s);
}

size_t zen_load_balance_workspace(int64_t n, int64_t m, int dtype, int64_t capacity, int partitions) {
  if (n <= 0 || m <= 0 || capacity < 0) return 0;
  const size_t general = zen::plan_balance(nullptr, n, m, dtype, capacity).bytes;
  const size_t slabs = partitions > 0 && m % partitions == 0 ? zen::slab_balance_bytes(m, partitions, dtype, capacity) : 0;
  const size_t wide = partitions > 0 && m % partitions == 0
                          ? zen::wide_balance_bytes(m, partitions, dtype, capacity, zen::wide_device_cus())
                          : 0;
  const size_t table = partitions > 0 && m % partitions == 0 ? zen::table_balance_bytes(n, m, dtype, partitions, capacity) : 0;
  const size_t buckets = slabs > wide ? slabs : wide;
  const size_t fast = buckets > table ? buckets : table;
  return general > fast ? general : fast;
}

}  // extern "C"

namespace {

// Whether a call takes the wide buckets where both they and the bucket slabs fit.  The resident kernel of the wide
// buckets is one launch where the slabs need four, but every workgroup of a partition looks at all of the partition's
// collisions; the slabs' chains share them out over the chip.  A call that waits for its sizes has the host idle: the
// slabs, which know the sizes before the entries are in place, are the quicker (compress and load balance of the top 1 %,
// us, wide and slabs: 4.3 M bf16 elements on 2 partitions 131 and 128; 8 M fp32 on 16 166 and 162; 36 M bf16 on 2 193 and
// 181; the hook on 130 M fp32 elements, 4 ranks, 596 and 570; densely the more, a load balance of 36 M with 10 % 714 and
// 166).  Calls that do not wait follow each other as fast as the host enqueues them, and the wide buckets are the quicker
// while collisions are few, up to about 8192 of them or one slot in 64 taken (three steps of 16 M bf16 elements on 16
// partitions with their merges, top 0.5 % 228 and 259, 2 % 259 and 273, 3.5 % 297 and 300, 5 % 350 and 325; of 36 M, 2 %
// 306 and 311, 3 % 383 and 343, 5 % 554 and 417; one of 743 M, 0.5 %, 392 and 493; three of 20 M with 0.5 % in whole rows,
// no threshold, 192 and 215).  asked: ZEN_MODE_WIDE.
bool takes_wide(int64_t n, int64_t m, int partitions, int dtype, int64_t capacity, int64_t k, bool waits, bool asked) {
  using namespace zen;
  if (!wide_balance_fits(m, partitions, capacity, k, wide_device_cus(), nullptr)) return false;
  if (asked) return true;
  const int64_t most = k > 0 ? k : capacity;
  const bool few = most <= m / 64 || (double)most * (double)most <= 2.0 * 8192.0 * (double)m;
  return (few && !waits) || !slab_balance_fits(n, m, partitions, dtype, capacity, k, nullptr);
}

}  // namespace

extern "C" {

int zen_load_balance_path(int64_t n, int64_t m, int dtype, int64_t capacity, int partitions, int64_t k, int mode) {
  const bool slabs_only = (mode & ZEN_MODE_SLABS) != 0, no_samples = (mode & ZEN_MODE_NO_SAMPLES) != 0;
  const bool ask_wide = (mode & ZEN_MODE_WIDE) != 0;
  mode &= 0xff;
  if (mode != ZEN_MODE_FAST || partitions <= 0 || m <= 0 || m % partitions != 0) return 0;
  const bool wide = !slabs_only && takes_wide(n, m, partitions, dtype, capacity, k, false, ask_wide);
  if (!slabs_only && !(wide && ask_wide) && zen::table_balance_fits(n, m, partitions, capacity, k, no_samples)) return 1;
  if (wide) return 3;
  if (zen::slab_balance_fits(n, m, partitions, dtype, capacity, k, nullptr)) return 2;
  return m >= 4096 ? 1 : 0;
}

namespace {

// the head of the table belongs to the hash map; the megabyte behind it is left to the slab path's counters
uint32_t slab_hash_log2(int64_t m) {
  uint32_t log2 = 0;
  while (log2 < 24 && (16ull << log2) + (1ull << 20) <= (uint64_t)m * sizeof(int32_t)) ++log2;
  return log2;
}

}  // namespace

int zen_load_balance_prepare(const void *input, int dtype, int64_t n, int64_t m, int partitions, int64_t k,
                             int64_t capacity, int32_t *table, int mode, void *workspace, size_t workspace_bytes,
                             void *stream) {
  using namespace zen;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_load_balance_prepare: bad dtype");
  if (n <= 0 || n > 0x7fffffffll || m <= 0 || m > 0x7fffffffll || partitions <= 0 || partitions > 65535 ||
      m % partitions != 0 || capacity <= 0 || capacity > 0x1fffffffll || k < 0 || k > n)
    return fail(ZEN_EINVAL, "zen_load_balance_prepare: sizes as for zen_load_balance");
  if (!input || !table || !workspace) return fail(ZEN_EINVAL, "zen_load_balance_prepare: null pointer");
  if (workspace_bytes < zen_load_balance_workspace(n, m, dtype, capacity, partitions))
    return fail(ZEN_EWORKSPACE, "zen_load_balance_prepare: workspace too small");
  const int second = (mode & ZEN_MODE_SECOND) != 0;
  if ((mode & 0xff) != ZEN_MODE_FAST || k == 0 || (reinterpret_cast<uintptr_t>(table) & 7u) != 0 ||
      (!(mode & ZEN_MODE_SLABS) && table_balance_fits(n, m, partitions, capacity, k, false)) ||
      (!slab_balance_fits(n, m, partitions, dtype, capacity, k, nullptr) &&
       !wide_balance_fits(m, partitions, capacity, k, wide_device_cus(), nullptr)))
    return ZEN_OK;  // nothing to take ahead on the other paths
  SlabBalanceArgs sa{};
  sa.input = input;
  sa.dtype = dtype;
  sa.n = n;
  sa.g.m = (uint32_t)m;
  sa.g.npp = (uint32_t)(m / partitions);
  sa.g.levels = 3;
  sa.partitions = partitions;
  sa.k = k;
  sa.capacity = capacity;
  sa.hash = reinterpret_cast<unsigned long long *>(table);
  sa.hash_log2 = slab_hash_log2(m);
  sa.workspace = workspace;
  sa.prepared = second ? 2 : 1;
  sa.second = second != 0;
  sa.only_prepare = true;
  sa.discard = (mode & ZEN_MODE_DISCARD) != 0;
  return slab_prepare(sa, static_cast<hipStream_t>(stream));
}

}  // extern "C"

namespace {

// zen_load_balance, and for zen_encode_merge the same with the next call's tensor handed along.
int load_balance_call(const void *input, int dtype, int64_t n, int64_t m, int partitions, int rehash,
                      const uint32_t *thr, int64_t k, uint32_t *thr_out, int32_t *out_idx, void *out_val,
                      int64_t capacity, int64_t *splits, int32_t *table, int mode, void *workspace,
                      size_t workspace_bytes, int32_t *status, void *stream, const void *next_input, int64_t next_k,
                      int64_t next_n, int64_t next_m, int64_t next_capacity, int32_t *next_table,
                      const zen::HostAsk &ask = {}) {
  using namespace zen;
  const int prepared = (mode & ZEN_MODE_PREPARED) ? ((mode & ZEN_MODE_SECOND) ? 2 : 1) : 0;
  const bool second_set = (mode & ZEN_MODE_SECOND) != 0;
  const uint32_t *near_key = nullptr;
  if (mode & ZEN_MODE_FLOOR) {
    if (k <= 0 || !thr) return fail(ZEN_EINVAL, "zen_load_balance: ZEN_MODE_FLOOR needs k > 0 and the key in thr");
    near_key = thr;
    thr = nullptr;  // paths that take no sample have no use for it
  }
  const bool slabs_only = (mode & ZEN_MODE_SLABS) != 0;
  const bool splits_zero = (mode & ZEN_MODE_ZEROED) != 0;
  const bool no_samples = (mode & ZEN_MODE_NO_SAMPLES) != 0;
  const bool ask_wide = (mode & ZEN_MODE_WIDE) != 0;
  mode &= ~(ZEN_MODE_PREPARED | ZEN_MODE_SECOND | ZEN_MODE_FLOOR | ZEN_MODE_SLABS | ZEN_MODE_ZEROED | ZEN_MODE_NO_SAMPLES |
            ZEN_MODE_WIDE);
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_load_balance: bad dtype");
  if (mode != ZEN_MODE_FAST && mode != ZEN_MODE_GENERAL) return fail(ZEN_EINVAL, "zen_load_balance: bad mode");
  if (n <= 0 || n > 0x7fffffffll || m <= 0 || m > 0x7fffffffll || partitions <= 0 || partitions > 65535 ||
      m % partitions != 0 || capacity <= 0 || capacity > 0x1fffffffll)
    return fail(ZEN_EINVAL, "zen_load_balance: need 0 < n, m < 2^31, m a multiple of partitions, 0 < capacity < 2^29");
  if (k < 0 || k > n || (k > 0 && thr)) return fail(ZEN_EINVAL, "zen_load_balance: need 0 <= k <= n and no thr with k");
  if (!input || !out_idx || !out_val || !splits || !table || !workspace || !status)
    return fail(ZEN_EINVAL, "zen_load_balance: null pointer");
  if (workspace_bytes < zen_load_balance_workspace(n, m, dtype, capacity, partitions))
    return fail(ZEN_EWORKSPACE, "zen_load_balance: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  Probe g;
  g.m = (uint32_t)m;
  g.npp = (uint32_t)(m / partitions);
  g.levels = (rehash == 2 || rehash == 3) ? rehash : 1;
  const int64_t spp = n / partitions / 10;  // tensor_load_balance.py:18
  const uint32_t drop_key = (uint32_t)partitions * (g.npp + 1u);
  const int bits = ceil_log2_u64(drop_key);
  const bool wide = mode == ZEN_MODE_FAST && !slabs_only && (reinterpret_cast<uintptr_t>(table) & 7u) == 0 &&
                    takes_wide(n, m, partitions, dtype, capacity, k, ask.answer.host != nullptr, ask_wide);
  const bool small = mode == ZEN_MODE_FAST && !slabs_only && !(wide && ask_wide) &&
                     (reinterpret_cast<uintptr_t>(table) & 15u) == 0 &&
                     table_balance_fits(n, m, partitions, capacity, k, no_samples);
  if (small || wide || (mode == ZEN_MODE_FAST && (reinterpret_cast<uintptr_t>(table) & 7u) == 0 &&
               slab_balance_fits(n, m, partitions, dtype, capacity, k, nullptr))) {
    SlabBalanceArgs sa;
    sa.input = input;
    sa.dtype = dtype;
    sa.n = n;
    sa.g = g;
    sa.partitions = partitions;
    sa.spp = spp;
    sa.thr = thr;
    sa.k = k;
    sa.thr_out = thr_out;
    sa.out_idx = out_idx;
    sa.out_val = out_val;
    sa.capacity = capacity;
    sa.splits = splits;
    sa.hash = reinterpret_cast<unsigned long long *>(table);
    sa.hash_log2 = slab_hash_log2(m);
    sa.workspace = workspace;
    sa.status = status;
    sa.prepared = near_key ? 0 : prepared;
    sa.second = second_set;
    sa.near_key = near_key;
    sa.ask = ask;
    if (small) return table_load_balance(sa, splits_zero, s);
    if (next_input && next_k > 0) {
      sa.next_input = next_input;
      sa.next_k = next_k;
      if (next_n > 0 || next_m > 0 || next_capacity > 0 || next_table) {  // a next call of its own size
        const int64_t n2 = next_n > 0 ? next_n : n, m2 = next_m > 0 ? next_m : m;
        const int64_t cap2 = next_capacity > 0 ? next_capacity : capacity;
        int32_t *table2 = next_table ? next_table : table;
        if (n2 > 0x7fffffffll || m2 > 0x7fffffffll || m2 % partitions != 0 || cap2 > 0x1fffffffll || next_k > n2 ||
            (reinterpret_cast<uintptr_t>(table2) & 7u) != 0 ||
            (!(!slabs_only && wide_balance_fits(m2, partitions, cap2, next_k, wide_device_cus(), nullptr)) &&
             !slab_balance_fits(n2, m2, partitions, dtype, cap2, next_k, nullptr)))  // (with this call's ZEN_MODE_SLABS)
          return fail(ZEN_EINVAL, "zen_encode_merge: the next call's sizes do not take a path that keeps a sample");
        if (workspace_bytes < zen_load_balance_workspace(n2, m2, dtype, cap2, partitions))
          return fail(ZEN_EWORKSPACE, "zen_encode_merge: workspace too small for the next call");
        sa.next_n = n2;
        sa.next_state = reinterpret_cast<char *>(table2) + slab_state_offset(slab_hash_log2(m2));
      }
    }
    if (wide) return wide_load_balance(sa, slab_state_offset(sa.hash_log2), s);
    return slab_load_balance(sa, s);
  }
  BalancePlan p = plan_balance(workspace, n, m, dtype, capacity);

  const uint32_t *filter = nullptr;
  int rc = select_stage(p, input, dtype, n, thr, k, capacity, mode, &filter, status, s);
  if (rc != ZEN_OK) return rc;
  if (k > 0 && thr_out) ZEN_HIP_CHECK(hipMemcpyAsync(thr_out, p.thr, 2 * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
  const int64_t lcap = list_capacity(capacity);
  if (mode == ZEN_MODE_FAST && m >= 4096 && (reinterpret_cast<uintptr_t>(table) & 7u) == 0) {
    // sort-based resolution: the table only lends its (zero) memory to a small hash map
    ResolveArgs ra;
    ra.dense = input;
    ra.dtype = dtype;
    ra.g = g;
    ra.partitions = partitions;
    ra.spp = spp;
    ra.list_idx = p.sel_idx;
    ra.list_val = p.sel_val;
    ra.count = p.count;
    ra.filter = filter;
    ra.list_cap = lcap;
    ra.expected = k > 0 ? k + k / 16 + 1024 : capacity;
    ra.keys_a = p.keys_a;
    ra.perm_a = p.perm_a;
    ra.keys_b = p.keys_b;
    ra.perm_b = p.perm_b;
    ra.more_a = p.more_a;
    ra.more_b = p.more_b;
    ra.sort_scratch = p.sort_scratch;
    ra.hash = reinterpret_cast<unsigned long long *>(table);
    uint32_t log2 = 0;
    while (log2 < 24 && (2ull << log2) <= (uint64_t)m / 2) ++log2;
    ra.hash_log2 = log2;
    ra.scratch = p.resolve_scratch;
    ra.out_idx = out_idx;
    ra.out_val = out_val;
    ra.capacity = capacity;
    ra.splits = splits;
    ra.status = status;
    return resolve_and_place(ra, s);
  }
  const unsigned blocks = (unsigned)ceil_div(lcap, 256);
  uint32_t *tab = reinterpret_cast<uint32_t *>(table);
  const uint16_t *val16 = reinterpret_cast<const uint16_t *>(p.sel_val);
  {
    ProfScope prof(kProfInsertList, s);
    if (dtype == ZEN_BF16)
      k_insert_list<uint16_t><<<dim3(blocks), dim3(256), 0, s>>>(p.sel_idx, val16, p.count, filter, tab, g);
    else
      k_insert_list<uint32_t><<<dim3(blocks), dim3(256), 0, s>>>(p.sel_idx, p.sel_val, p.count, filter, tab, g);
    ZEN_LAUNCH_CHECK("k_insert_list");
  }
  {
    ProfScope prof(kProfFinalKey, s);
    if (dtype == ZEN_BF16)
      k_final_key<uint16_t><<<dim3(blocks), dim3(256), 0, s>>>(p.sel_idx, val16, p.count, filter, tab, g, drop_key,
                                                               p.keys_a, p.perm_a);
    else
      k_final_key<uint32_t><<<dim3(blocks), dim3(256), 0, s>>>(p.sel_idx, p.sel_val, p.count, filter, tab, g, drop_key,
                                                               p.keys_a, p.perm_a);
    ZEN_LAUNCH_CHECK("k_final_key");
  }
  int where;
  {
    ProfScope prof(kProfSort, s);
    where = sort_pairs(p.keys_a, p.perm_a, p.keys_b, p.perm_b, lcap, p.count, bits, p.sort_scratch, status, s);
  }
  if (where < 0) return where;
  const uint32_t *sk = where ? p.keys_b : p.keys_a;
  const uint32_t *sp = where ? p.perm_b : p.perm_a;
  {
    ProfScope prof(kProfGather, s);
    if (dtype == ZEN_BF16)
      k_gather<uint16_t><<<dim3(blocks), dim3(256), 0, s>>>(sk, sp, p.count, p.sel_idx, val16, drop_key, g, out_idx,
                                                            static_cast<uint16_t *>(out_val), (uint32_t)capacity, tab);
    else
      k_gather<uint32_t><<<dim3(blocks), dim3(256), 0, s>>>(sk, sp, p.count, p.sel_idx, p.sel_val, drop_key, g, out_idx,
                                                            static_cast<uint32_t *>(out_val), (uint32_t)capacity, tab);
    ZEN_LAUNCH_CHECK("k_gather");
  }
  if (dtype == ZEN_BF16)
    k_splits_serial<uint16_t><<<dim3((unsigned)partitions), dim3(256), 0, s>>>(
        sk, p.count, g.npp, spp, (uint32_t)capacity, static_cast<const uint16_t *>(input), out_idx,
        static_cast<uint16_t *>(out_val), splits, status);
  else
    k_splits_serial<uint32_t><<<dim3((unsigned)partitions), dim3(256), 0, s>>>(
        sk, p.count, g.npp, spp, (uint32_t)capacity, static_cast<const uint32_t *>(input), out_idx,
        static_cast<uint32_t *>(out_val), splits, status);
  ZEN_LAUNCH_CHECK("k_splits_serial");
  return ZEN_OK;
}

}  // namespace

extern "C" {

int zen_load_balance(const void *input, int dtype, int64_t n, int64_t m, int partitions, int rehash,
                     const uint32_t *thr, int64_t k, uint32_t *thr_out, int32_t *out_idx, void *out_val,
                     int64_t capacity, int64_t *splits, int32_t *table, int mode, void *workspace,
                     size_t workspace_bytes, int32_t *status, void *stream) {
  return load_balance_call(input, dtype, n, m, partitions, rehash, thr, k, thr_out, out_idx, out_val, capacity, splits,
                           table, mode, workspace, workspace_bytes, status, stream, nullptr, 0, 0, 0, 0, nullptr);
}

int zen_load_balance_sizes(const void *input, int dtype, int64_t n, int64_t m, int partitions, int rehash,
                           const uint32_t *thr, int64_t k, uint32_t *thr_out, int32_t *out_idx, void *out_val,
                           int64_t capacity, int64_t *splits, int32_t *table, int mode, void *workspace,
                           size_t workspace_bytes, int32_t *status, int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  bool answered = false;
  int rc = host_ask(host, words, (int64_t)partitions + 1, &answer);
  if (rc != ZEN_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = load_balance_call(input, dtype, n, m, partitions, rehash, thr, k, thr_out, out_idx, out_val, capacity, splits, table,
                         mode, workspace, workspace_bytes, status, stream, nullptr, 0, 0, 0, 0, nullptr, HostAsk{answer, &answered});
  if (rc == ZEN_OK && !answered) rc = host_answer_launch(answer, splits, partitions, status, 1, s);
  return host_finish(rc, answer, s);
}

int zen_encode_merge_samples_next(int64_t n, int64_t m, int dtype, int64_t capacity, int partitions, int64_t k,
                                  int mode) {
  const int path = zen_load_balance_path(n, m, dtype, capacity, partitions, k, mode);
  return path == 2 || path == 3;
}

int zen_encode_merge(const zen_encode_merge_args *a) {
  using namespace zen;
  if (!a) return fail(ZEN_EINVAL, "zen_encode_merge: null pointer");
  const int rc = load_balance_call(a->input, a->dtype, a->n, a->m, a->partitions, a->rehash, a->thr, a->k, a->thr_out,
                                   a->out_idx, a->out_val, a->capacity, a->splits, a->table, a->mode, a->workspace,
                                   a->workspace_bytes, a->status, a->stream, a->next_input, a->next_k, a->next_n,
                                   a->next_m, a->next_capacity, a->next_table);
  if (rc != ZEN_OK) return rc;
  return zen_merge(a->recv_idx, a->recv_idx64, a->recv_val, a->dtype, a->r, a->dense_n, a->merged_idx, a->merged_idx64,
                   a->merged_val, a->merged_capacity, a->merged_count, a->merge_mode, a->merge_workspace,
                   a->merge_workspace_bytes, a->merge_status, a->merge_stream ? a->merge_stream : a->stream);
}

}  // extern "C"
