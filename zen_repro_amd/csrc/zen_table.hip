// Fused load balance through the owner table, for small inputs.
//
// What the reference does (functions_cuda_kernel.cu:97-167, tensor_load_balance.py:13-51): every selected index goes
// into a hash table as large as the gradient, and the table, read in slot order, is the output.  For a few million
// slots at most that is also the quickest way: the table fits the caches, nothing has to be sorted, and the steps
// are few (the sort-based resolution took 23 launches, most of them waiting for the one before):
//   k_table_insert  selects while it reads the tensor and inserts with atomicMax on 0 - index (a slot belongs to the
//                   smallest index that ever probes it; who takes a slot from a larger index continues that index's
//                   probes, as in zen_balance.hip); an index that is out of levels takes a ticket of its partition's
//                   serial region;
//   k_table_out     entries in slot order to their places (every stretch of the table says how many it holds, and adds up
//                   what the ones before it said), serial tails, split sizes; empties the table again; tells the host.
// Up to kOneSlots slots the table is kept in LDS and one workgroup does all of it (k_table_one).
// Bound by latency.
#include "zen_balance.h"

namespace zen {
namespace {

constexpr int kInsBlock = 512;
constexpr int kOutBlock = 1024;
constexpr int kOutRows = 4;                                 // rows of 256 slots per wave
// Slots per workgroup: 16 384.  A workgroup draws a ticket, adds to a partition's size and counts itself as finished, all
// on lines that take ten nanoseconds each time: with stretches of 4096 (256 threads) 4.1 M slots took 87 us, now 70.
constexpr uint32_t kStretch = kOutBlock / 64 * kOutRows * 256;
constexpr int kMaxParts = 1024;
constexpr int kOneBlock = 1024;
constexpr uint32_t kOneSlots = 32768;                       // 128 KB of LDS
constexpr int kOneParts = 256;
constexpr uint32_t kOneList = 4096;                         // selected indices side by side
constexpr uint32_t kOneSerial = 3456;                       // more than a tenth of kOneSlots: more would be an overflow

// Inserts index t.  Returns the index that ends up without a slot (0: none) and its partition.
__device__ inline uint32_t insert(uint32_t *table, const Probe &g, uint32_t t, uint32_t *part) {
  uint32_t cur = t;
  int lv = 0;
  for (;;) {
    const uint32_t slot = probe_slot(g, cur, lv, part);
    const uint32_t mine = 0u - cur;
    const uint32_t old = atomicMax(&table[slot], mine);
    if (old > mine) {  // a smaller index owns the slot: cur moves on
      if (++lv >= g.levels) return cur;
      continue;
    }
    if (old == 0u || old == mine) return 0;
    // took the slot from a larger index, which goes on behind its first level that maps here
    cur = 0u - old;
    lv = 0;
    while (lv < g.levels && probe_slot(g, cur, lv, part) != slot) ++lv;
    if (++lv >= g.levels) return cur;
  }
}

__device__ inline uint32_t least_key(const uint32_t *thr, uint32_t mask) {
  uint32_t t = thr ? thr[0] : 1u;
  if (t == 0) t = 1;
  return t > mask ? mask + 1u : t;
}

struct Tables {
  uint32_t *slots;       // [m] the caller's table, zero between calls
  unsigned long long *splits;  // [P], zero: serial tickets in the upper halves while the indices are inserted
  uint32_t *serial;      // [P * ser_cap] indices without a slot
  unsigned long long *desc;  // [stretches] entries each holds, and behind them the words of `ticket` and `done`
  uint32_t *ticket, *done;   // stretches taken, stretches finished
  uint32_t ser_cap;
  int parts;
  int64_t spp;           // serial slots of the reference's table, per partition
};

// Indices of partition p without a slot, as long as its tickets are in the upper half of its split size.
__device__ inline uint32_t tickets(const Tables &tb, int p) {
  const uint32_t s = (uint32_t)(__hip_atomic_load(&tb.splits[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 32);
  return s < tb.ser_cap ? s : tb.ser_cap;
}

template <typename S, bool ALIGNED>
__global__ __launch_bounds__(kInsBlock) void k_table_insert(const S *__restrict__ in, int64_t n,
                                                            const uint32_t *__restrict__ thr, Probe g, Tables tb,
                                                            uint32_t stretches, int32_t *status) {
  // the selected indices of the workgroup's stretch side by side, so that every thread has one to insert
  constexpr int V = VecOf<S>::kN;
  __shared__ uint32_t list[kInsBlock * V];
  __shared__ uint32_t count;
  if (threadIdx.x == 0) count = 0;
  for (uint32_t i = blockIdx.x * kInsBlock + threadIdx.x; i <= stretches; i += gridDim.x * kInsBlock) tb.desc[i] = 0ull;
  const uint32_t least = least_key(thr, KeyOf<S>::kMask);
  const int64_t first = ((int64_t)blockIdx.x * kInsBlock + threadIdx.x) * V;
  S e[V];
  load_vec<S, ALIGNED>(in, first, n, e);
  uint32_t flags = 0;
#pragma unroll
  for (int i = 0; i < V; ++i) flags |= (uint32_t)((uint32_t)(e[i] & KeyOf<S>::kMask) >= least) << i;
  if (first == 0) flags &= ~1u;  // index 0 is never transmitted
  const uint32_t c = (uint32_t)__popc(flags);
  const uint32_t incl = wave_inclusive_scan(c);
  __syncthreads();
  uint32_t at = 0;
  if (lane_id() == 63 && incl) at = atomicAdd(&count, incl);
  at = (uint32_t)__builtin_amdgcn_readlane((int)at, 63) + incl - c;
  while (flags) {
    list[at++] = (uint32_t)first + (uint32_t)__ffs((int)flags) - 1u;
    flags &= flags - 1u;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < count; i += kInsBlock) {
    uint32_t part;
    const uint32_t left = insert(tb.slots, g, list[i], &part);
    if (left) {
      const uint32_t ticket = (uint32_t)(atomicAdd(&tb.splits[part], 1ull << 32) >> 32);
      if ((int64_t)ticket >= tb.spp) atomicOr(status, ZEN_STAT_SERIAL_OVERFLOW);
      if (ticket < tb.ser_cap) tb.serial[(size_t)part * tb.ser_cap + ticket] = left;
    }
  }
}

// The slots [base, base + 4) of lane `lane` in row r of the wave, those past the table as empty.
__device__ inline uint4 load_slots(const uint32_t *slots, uint32_t at, uint32_t m) {
  if (at + 4 <= m) return *reinterpret_cast<const uint4 *>(slots + at);
  uint4 q = make_uint4(0, 0, 0, 0);
  if (at < m) q.x = slots[at];
  if (at + 1 < m) q.y = slots[at + 1];
  if (at + 2 < m) q.z = slots[at + 2];
  return q;
}
__device__ inline uint32_t occupied(const uint4 &q) {
  return (q.x ? 1u : 0u) | (q.y ? 2u : 0u) | (q.z ? 4u : 0u) | (q.w ? 8u : 0u);
}
__device__ inline uint32_t word_of(const uint4 &q, uint32_t e) {
  const uint32_t a = e & 1u ? q.y : q.x, b = e & 1u ? q.w : q.z;
  return e & 2u ? b : a;
}

// Bound by the trips to memory: the slots, what the stretches before hold, the entries' values, the host.  The entries
// are put side by side in LDS first, so that all of a stretch's values are on their way together (each thread's own
// entries one after the other: 12 us for 145 000 bf16 slots, 10 % taken); with a kernel for the counts in front and one for
// the host behind, a load balance of 300 000 bf16 elements took 46 us, of 2.2 M, 10 % selected, 74.
template <typename S>
__global__ __launch_bounds__(kOutBlock) void k_table_out(const S *__restrict__ dense, Tables tb, uint32_t m, uint32_t npp,
                                                         uint32_t stretches, int32_t *__restrict__ out_idx,
                                                         S *__restrict__ out_val, uint32_t capacity, HostAnswer answer,
                                                         int32_t *status) {
  __shared__ uint32_t smem[kOutBlock / 64 + 1];
  __shared__ uint32_t before_part[kMaxParts + 1];  // serial entries of the partitions before
  __shared__ uint32_t buf[kStretch + kMaxParts];   // the stretch's entries and its partitions' counts, then a serial tail
  __shared__ uint32_t ends_at[kOutBlock];
  __shared__ uint32_t s_turn;
  static_assert(kSerialLds <= kStretch + kMaxParts, "room for a tail");
  uint32_t *held = buf + kStretch;
  if (threadIdx.x == 0) s_turn = atomicAdd(tb.ticket, 1u);
  __syncthreads();
  const uint32_t c = s_turn;  // stretches are taken in order, so every earlier one already runs
  if (c >= stretches) return;
  const uint32_t wave = threadIdx.x >> 6, lane = (uint32_t)lane_id();
  const uint32_t base = c * kStretch + wave * (kOutRows * 256) + lane * 4;
  uint4 q[kOutRows];
#pragma unroll
  for (int r = 0; r < kOutRows; ++r) q[r] = load_slots(tb.slots, base + r * 256, m);
  // The stretch's partitions, p_first to p_last.  Where it has several, their entries are counted in LDS (an add to the
  // split sizes for every entry of such a stretch: some 6000 of them queue on one line, 1.8 M fp32 slots, 5 % taken, 16
  // partitions 27 us, then 8).
  const uint32_t lo = c * kStretch, hi = lo + kStretch < m ? lo + kStretch : m;  // lo < m
  const uint32_t p_first = lo / npp, p_last = (hi - 1u) / npp;
  if (p_first != p_last)
    for (uint32_t i = threadIdx.x; i <= p_last - p_first; i += kOutBlock) held[i] = 0;
  uint32_t mine = 0;
#pragma unroll
  for (int r = 0; r < kOutRows; ++r) mine += (uint32_t)__popc(occupied(q[r]));
  const uint32_t in_wave = wave_sum(mine);
  if (lane == 0) smem[wave] = in_wave;
  __syncthreads();
  uint32_t at = 0, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < kOutBlock / 64; ++w) {
    at += w < wave ? smem[w] : 0u;
    all += smem[w];
  }
  if (threadIdx.x == 0) desc_store(&tb.desc[c], kDescAggregate | all);
#pragma unroll
  for (int r = 0; r < kOutRows; ++r) {
    const uint32_t x = occupied(q[r]);
    const uint32_t n = (uint32_t)__popc(x), incl = wave_inclusive_scan(n);
    uint32_t pos = at + incl - n;
    for (uint32_t bits = x; bits; bits &= bits - 1u, ++pos) buf[pos] = 0u - word_of(q[r], (uint32_t)__ffs((int)bits) - 1u);
    at += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    if (x) {  // leave the table empty again
      const uint32_t s0 = base + r * 256;
      if (s0 + 4 <= m) {
        *reinterpret_cast<uint4 *>(tb.slots + s0) = make_uint4(0, 0, 0, 0);
      } else {
        for (uint32_t i = 0; s0 + i < m; ++i) tb.slots[s0 + i] = 0;
      }
    }
  }
  // entries in front of the stretch (bounded waits), and serial entries in front of every partition
  uint32_t sum = 0, front;
  for (uint32_t i = threadIdx.x; i < c; i += kOutBlock) {
    uint64_t d = desc_load(&tb.desc[i]);
    uint32_t spins = 0;
    while ((d >> 62) == 0) {
      if (++spins > kSpinLimit) {
        atomicOr(status, ZEN_STAT_INTERNAL);
        break;
      }
      __builtin_amdgcn_s_sleep(2);
      d = desc_load(&tb.desc[i]);
    }
    sum += (uint32_t)(d & kDescValue);
  }
  __syncthreads();  // (smem has been read)
  block_exclusive_scan<uint32_t, kOutBlock>(sum, smem, &front);
  uint32_t carry = 0;
  for (int p0 = 0; p0 < tb.parts; p0 += kOutBlock) {
    const int p = p0 + (int)threadIdx.x;
    const uint32_t s = p < tb.parts ? tickets(tb, p) : 0u;
    uint32_t total;
    const uint32_t ex = block_exclusive_scan<uint32_t, kOutBlock>(s, smem, &total);
    if (p < tb.parts) before_part[p] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) before_part[tb.parts] = carry;
  __syncthreads();
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < all; i += kOutBlock) {
    const uint32_t t = buf[i];
    uint32_t p = p_first;
    if (p_first != p_last) {  // (an index stays in the partition of its first slot)
      p = (poly(t) + kSeed1) % m / npp;
      atomicAdd(&held[p - p_first], 1u);
    }
    const uint32_t to = front + i + before_part[p];
    if (to < capacity) {
      out_idx[to] = (int32_t)t;
      out_val[to] = dense[t];
    }
  }
  if (p_first == p_last) {
    if (threadIdx.x == 0 && all) atomicAdd(&tb.splits[p_first], (unsigned long long)all);
  } else {
    __syncthreads();
    for (uint32_t i = threadIdx.x; i <= p_last - p_first; i += kOutBlock)
      if (held[i]) atomicAdd(&tb.splits[p_first + i], (unsigned long long)held[i]);
  }
  if (c == stretches - 1 && threadIdx.x == 0 && front + all + carry > capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  // the serial tails of the partitions that end in this stretch, in ascending index order
  for (uint32_t p = p_first; p <= p_last; ++p) {
    const uint32_t end = (p + 1u) * npp;  // <= m
    const uint32_t n = before_part[p + 1] - before_part[p];
    if (end > hi || n == 0) continue;  // (uniform)
    // entries of the stretch in front of the partition's end
    uint32_t in_front = 0;
#pragma unroll
    for (int r = 0; r < kOutRows; ++r) {
      const uint32_t s0 = base + r * 256;
      const uint32_t keep = s0 >= end ? 0u : end - s0 >= 4u ? 15u : (1u << (end - s0)) - 1u;
      in_front += (uint32_t)__popc(occupied(q[r]) & keep);
    }
    uint32_t total;
    __syncthreads();
    block_exclusive_scan<uint32_t, kOutBlock>(in_front, ends_at, &total);
    const uint32_t to = front + total + before_part[p];
    if (to + n <= capacity) {
      for (uint32_t i = threadIdx.x; i < n; i += kOutBlock) {
        out_idx[to + i] = (int32_t)tb.serial[(size_t)p * tb.ser_cap + i];
        out_val[to + i] = dense[tb.serial[(size_t)p * tb.ser_cap + i]];
      }
      __syncthreads();
      fix_serial_tail<S>(out_idx, out_val, dense, to, n, buf);
      __syncthreads();
    }
  }
  // the stretch that finishes last turns tickets and counts into the split sizes
  wait_global_acks();
  __syncthreads();
  if (threadIdx.x == 0) s_turn = atomicAdd(tb.done, 1u);
  __syncthreads();
  if (s_turn != stretches - 1u) return;
  for (int p = threadIdx.x; p < tb.parts; p += kOutBlock) {
    const unsigned long long both = __hip_atomic_load(&tb.splits[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int64_t size = (int64_t)(both & 0xffffffffull) + (int64_t)tickets(tb, p);
    tb.splits[p] = (unsigned long long)size;
    if (answer.host) host_store(answer.host + 1 + p, size);
  }
  if (answer.host) {
    if (threadIdx.x == 0)
      host_store(answer.host + 1 + tb.parts, (int64_t)__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    host_answered(answer);
  }
}

template <typename S, bool ALIGNED>
__global__ __launch_bounds__(kOneBlock) void k_table_one(const S *__restrict__ in, uint32_t n,
                                                         const uint32_t *__restrict__ thr, Probe g, int parts, int64_t spp,
                                                         int32_t *__restrict__ out_idx, S *__restrict__ out_val,
                                                         uint32_t capacity, int64_t *__restrict__ splits,
                                                         HostAnswer answer, int32_t *status) {
  constexpr int V = VecOf<S>::kN;
  __shared__ __attribute__((aligned(16))) uint32_t slots[kOneSlots];
  __shared__ uint32_t serial[kOneSerial];       // partition << 15 | index
  __shared__ uint32_t held[kOneParts], left[kOneParts], before_left[kOneParts];
  __shared__ uint32_t smem[kOneBlock / 64 + 1];
  __shared__ uint16_t list[kOneList];
  __shared__ uint32_t serial_n;
  const uint32_t m = g.m;
  const uint32_t words = (m + 3u) / 4u * 4u;
  for (uint32_t i = threadIdx.x * 4; i < words; i += kOneBlock * 4) *reinterpret_cast<uint4 *>(slots + i) = make_uint4(0, 0, 0, 0);
  if (threadIdx.x < kOneParts) held[threadIdx.x] = left[threadIdx.x] = 0;
  if (threadIdx.x == 0) serial_n = 0;
  const uint32_t least = least_key(thr, KeyOf<S>::kMask);
  // All of the tensor is asked for at once; then the selected indices side by side, so that every thread has one to insert
  // (9219 bf16 elements, 10 % selected: 16 us, 7.7 of them here, with a round of this for every 4096 elements; 17.6 with
  // every thread inserting its own elements one after the other).
  constexpr int kRows = (int)(kOneSlots / (kOneBlock * V));
  uint32_t flags[kRows];
  uint32_t mine_n = 0;
  {
    S e[kRows][V];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const uint32_t first = ((uint32_t)r * kOneBlock + threadIdx.x) * V;
      if ((uint32_t)r * kOneBlock * V < n) load_vec<S, ALIGNED>(in, first, n, e[r]);  // (places past the end: zeros)
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      flags[r] = 0;
      if ((uint32_t)r * kOneBlock * V < n) {
#pragma unroll
        for (int i = 0; i < V; ++i) flags[r] |= (uint32_t)((uint32_t)(e[r][i] & KeyOf<S>::kMask) >= least) << i;
      }
      if (r == 0 && threadIdx.x == 0) flags[r] &= ~1u;  // index 0 is never transmitted
      mine_n += (uint32_t)__popc(flags[r]);
    }
  }
  uint32_t selected;
  const uint32_t ahead = block_exclusive_scan<uint32_t, kOneBlock>(mine_n, smem, &selected);  // (its barriers: the slots are empty)
  for (uint32_t from = 0; from < selected; from += kOneList) {
    uint32_t at = ahead;
#pragma unroll
    for (int r = 0; r < kRows; ++r)
      for (uint32_t bits = flags[r]; bits; bits &= bits - 1u, ++at)
        if (at - from < kOneList) list[at - from] = (uint16_t)(((uint32_t)r * kOneBlock + threadIdx.x) * V + (uint32_t)__ffs((int)bits) - 1u);
    __syncthreads();
    const uint32_t listed = selected - from < kOneList ? selected - from : kOneList;
    for (uint32_t i = threadIdx.x; i < listed; i += kOneBlock) {
      uint32_t part;
      const uint32_t out = insert(slots, g, list[i], &part);
      if (out) {
        const uint32_t place = atomicAdd(&serial_n, 1u);
        if (place < kOneSerial) {
          serial[place] = (part << 15) | out;
          atomicAdd(&left[part], 1u);
        } else {
          atomicOr(status, ZEN_STAT_SERIAL_OVERFLOW);  // some partition has more than its tenth
        }
      }
    }
    __syncthreads();
  }
  __syncthreads();
  const uint32_t total_left = serial_n < kOneSerial ? serial_n : kOneSerial;
  if (total_left > 1) sort_network(serial, total_left);
  {
    const uint32_t s = threadIdx.x < kOneParts ? left[threadIdx.x] : 0u;
    uint32_t total;
    const uint32_t ex = block_exclusive_scan<uint32_t, kOneBlock>(s, smem, &total);
    if (threadIdx.x < kOneParts) before_left[threadIdx.x] = ex;
    if ((int64_t)s > spp) atomicOr(status, ZEN_STAT_SERIAL_OVERFLOW);
  }
  // a wave's slots: a sixteenth of the table, in rows of 256
  const uint32_t wave = threadIdx.x >> 6, lane = (uint32_t)lane_id();
  const uint32_t rows = (m + 16 * 256 - 1) / (16 * 256);
  const uint32_t base = wave * rows * 256 + lane * 4;
  uint32_t mine = 0;
  for (uint32_t r = 0; r < rows; ++r) mine += (uint32_t)__popc(base + r * 256 < words ? occupied(*reinterpret_cast<const uint4 *>(slots + base + r * 256)) : 0u);
  const uint32_t in_wave = wave_sum(mine);
  __syncthreads();
  if (lane == 0) smem[wave] = in_wave;
  __syncthreads();
  uint32_t at = 0, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < kOneBlock / 64; ++w) {
    at += w < wave ? smem[w] : 0u;
    all += smem[w];
  }
  // a wave puts its entries side by side at the head of its own slots (which it has read by then), ...
  uint32_t put = 0;
  for (uint32_t r = 0; r < rows; ++r) {
    const uint32_t s0 = base + r * 256;
    const uint4 q = s0 < words ? *reinterpret_cast<const uint4 *>(slots + s0) : make_uint4(0, 0, 0, 0);
    const uint32_t x = occupied(q), c = (uint32_t)__popc(x), incl = wave_inclusive_scan(c);
    uint32_t pos = wave * rows * 256 + put + incl - c;
    __builtin_amdgcn_wave_barrier();  // (the row is read by all lanes before any of them writes)
    for (uint32_t bits = x; bits; bits &= bits - 1u, ++pos) slots[pos] = 0u - word_of(q, (uint32_t)__ffs((int)bits) - 1u);
    put += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
  }
  // ... and takes them to their places, all values on their way together
  for (uint32_t i = lane; i < in_wave; i += 64) {
    const uint32_t t = slots[wave * rows * 256 + i], p = (poly(t) + kSeed1) % m / g.npp;  // (it stays in its first slot's partition)
    atomicAdd(&held[p], 1u);
    const uint32_t to = at + i + before_left[p];
    if (to < capacity) {
      out_idx[to] = (int32_t)t;
      out_val[to] = in[t];
    }
  }
  __syncthreads();
  {
    const uint32_t h = threadIdx.x < kOneParts ? held[threadIdx.x] : 0u;
    uint32_t total;
    const uint32_t ex = block_exclusive_scan<uint32_t, kOneBlock>(h, smem, &total);
    if ((int)threadIdx.x < parts) {
      splits[threadIdx.x] = (int64_t)(h + left[threadIdx.x]);
      if (answer.host) host_store(answer.host + 1 + threadIdx.x, (int64_t)(h + left[threadIdx.x]));
    }
    if (threadIdx.x < kOneParts) held[threadIdx.x] = ex + h;  // entries with a slot through the partition
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total_left; i += kOneBlock) {
    const uint32_t t = serial[i] & 0x7fffu, to = held[serial[i] >> 15] + i;
    if (to < capacity) {
      out_idx[to] = (int32_t)t;
      out_val[to] = in[t];
    }
  }
  if (threadIdx.x == 0 && all + total_left > capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  if (answer.host) {
    wait_global_acks();
    __syncthreads();
    if (threadIdx.x == 0)
      host_store(answer.host + 1 + parts, (int64_t)__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    host_answered(answer);
  }
}

struct TablePlan {
  uint32_t *thr;
  Tables tb;
  void *topk;
  uint32_t stretches;
  size_t bytes;
};

TablePlan plan_table(void *workspace, int64_t n, int64_t m, int dtype, int partitions) {
  Carver cv(workspace);
  TablePlan p{};
  p.thr = cv.take<uint32_t>(2);
  p.stretches = (uint32_t)ceil_div(m, (int64_t)kStretch);
  const int64_t spp = n / partitions / 10;
  p.tb.ser_cap = (uint32_t)(spp > 64 ? spp : 64);
  p.tb.serial = cv.take<uint32_t>((size_t)p.tb.ser_cap * partitions);
  p.tb.desc = cv.take<unsigned long long>((size_t)p.stretches + 1);
  p.tb.ticket = reinterpret_cast<uint32_t *>(p.tb.desc + p.stretches);
  p.tb.done = p.tb.ticket + 1;
  p.topk = cv.take<char>(topk_whole_bytes(n, dtype));
  p.tb.parts = partitions;
  p.tb.spp = spp;
  p.bytes = cv.used;
  return p;
}

template <typename S, bool ALIGNED>
int table_launch(const SlabBalanceArgs &a, const TablePlan &p, const uint32_t *thr, bool zeroed, hipStream_t s) {
  const S *in = static_cast<const S *>(a.input);
  S *out_val = static_cast<S *>(a.out_val);
  if (a.g.m <= kOneSlots && a.n <= (int64_t)kOneSlots && a.partitions <= kOneParts) {
    k_table_one<S, ALIGNED><<<dim3(1), dim3(kOneBlock), 0, s>>>(in, (uint32_t)a.n, thr, a.g, a.partitions, a.spp, a.out_idx,
                                                               out_val, (uint32_t)a.capacity, a.splits, a.ask.answer,
                                                               a.status);
    ZEN_LAUNCH_CHECK("k_table_one");
    if (a.ask.answer.host) *a.ask.answered = true;
    return ZEN_OK;
  }
  if (!zeroed) launch_fill<int64_t>(a.splits, 0, (size_t)a.partitions, s);
  const int64_t blocks = ceil_div(a.n, (int64_t)kInsBlock * VecOf<S>::kN);
  k_table_insert<S, ALIGNED><<<dim3((unsigned)blocks), dim3(kInsBlock), 0, s>>>(in, a.n, thr, a.g, p.tb, p.stretches, a.status);
  ZEN_LAUNCH_CHECK("k_table_insert");
  k_table_out<S><<<dim3(p.stretches), dim3(kOutBlock), 0, s>>>(in, p.tb, a.g.m, a.g.npp, p.stretches, a.out_idx, out_val,
                                                              (uint32_t)a.capacity, a.ask.answer, a.status);
  ZEN_LAUNCH_CHECK("k_table_out");
  if (a.ask.answer.host) *a.ask.answered = true;
  return ZEN_OK;
}

}  // namespace

// A selection by a given threshold, or of the nonzeros: the atomics and two readings of the table cost less than the bucket
// slabs' five launches up to 6 Mi slots, up to 10 Mi where little is selected (a call that waits, 2 partitions, us here and
// on the slabs: 6 M bf16 elements 0.5 % selected 50 and 62, 5 % 67 and 74, 10 % 90 and 88; 9 M 58 and 63, 1.5 % 62 and 65,
// 5 % 85 and 77; 16 M 71 and 67, 5 % 113 and 90).  A top-k selection, whose threshold takes launches of its own here, only
// where the wide buckets do not apply.  Every word of the table is a slot here, and a sample taken ahead waits in its call's
// table, in tables of 2^20 slots or more (wide_geometry, slab_geometry): those are taken only if there is none, the others
// hold none.
bool table_balance_fits(int64_t n, int64_t m, int partitions, int64_t capacity, int64_t k, bool no_samples) {
  const int64_t most = k > 0 || !no_samples ? (1ll << 20) - 1 : capacity <= m / 32 ? 10ll << 20 : 6ll << 20;
  return n <= (10ll << 20) && m <= most && partitions <= kMaxParts;
}

size_t table_balance_bytes(int64_t n, int64_t m, int dtype, int partitions, int64_t capacity) {
  return table_balance_fits(n, m, partitions, capacity, 0, true) ? plan_table(nullptr, n, m, dtype, partitions).bytes : 0;
}

int table_load_balance(const SlabBalanceArgs &a, bool splits_zero, hipStream_t s) {
  TablePlan p = plan_table(a.workspace, a.n, a.g.m, a.dtype, a.partitions);
  p.tb.slots = reinterpret_cast<uint32_t *>(a.hash);
  p.tb.splits = reinterpret_cast<unsigned long long *>(a.splits);
  const uint32_t *thr = a.thr;
  if (a.k > 0) {
    uint32_t *to = a.thr_out ? a.thr_out : p.thr;
    const int rc = topk_whole(a.input, a.dtype, a.n, a.k, to, p.topk, s);
    if (rc != ZEN_OK) return rc;
    thr = to;
  }
  const bool aligned = (reinterpret_cast<uintptr_t>(a.input) & 15u) == 0;
  if (a.dtype == ZEN_BF16)
    return aligned ? table_launch<uint16_t, true>(a, p, thr, splits_zero, s) : table_launch<uint16_t, false>(a, p, thr, splits_zero, s);
  return aligned ? table_launch<uint32_t, true>(a, p, thr, splits_zero, s) : table_launch<uint32_t, false>(a, p, thr, splits_zero, s);
}

}  // namespace zen
