// The lists of a filled hash table or overflow region (zen_table_find, zen_table_gather; get_sub_sparse_tensors,
// tensor_load_balance.py:24-40): every partition's nonzero entries in slot order and the values they point at.
//
// Every partition is cut into stretches of equal length, one per wave, so that no stretch crosses a partition's
// edge and the split sizes are sums of whole stretches.  k_table_walk leaves a stretch's entries side by side in the
// workspace and its last workgroup tells the host the split sizes; once the host has made buffers of just that size,
// k_table_gather moves the entries there and fetches their values.
// Bound by the read of the table and by the random lines the values lie on.  16.7 M slots of 5 % filled, eight
// partitions, bf16: 21 + 18 us.
// A compaction to (position, entry) lists, a search for the partitions' edges and two library launches per
// partition for the values took 330 us there, in 35 launches instead of 4.
#include "zen_common.h"

namespace zen {
namespace {

constexpr int kBlock = 256;                // of the walking kernel: a stretch per wave
constexpr int kRows = 4;                   // rows of one 16-byte vector per lane in flight
constexpr int64_t kRow = 64 * 4;           // entries of a row
constexpr int64_t kStep = kRow * kRows;
constexpr int64_t kMaxStretches = 8192;    // 32 waves per compute unit
constexpr int kScanBlock = 1024;
constexpr int kMoveBlock = 256;

// Up to here the walk adds up the partitions' sizes while it runs and the gather finds its places from the stretches'
// counts; with more partitions one workgroup does both in between (16.7 M slots, eight partitions: walk 15.6, sizes
// and places 8.5, read-back for the host 2.5 us and two gaps between launches; now 21 in one, the call's table, lists
// and those of its overflow region together 203 -> 197 us).  The bound keeps the marks and the answer small; sums over
// the counts, at most 8192 of them up to here, would grow with the partitions.
constexpr int kMostMarked = ZEN_TABLE_SIZES_MOST;
constexpr int kMarkGroup = 32;             // workgroups that count themselves as finished in one word

struct TablePlan {
  int64_t per_part;  // slots of a partition
  int64_t len;       // slots of a stretch
  int64_t cpp;       // stretches of a partition
  int64_t count;     // stretches
  uint32_t *found;   // [count]
  uint32_t *at;      // [count + 1]
  int32_t *entries;  // [partitions * per_part], a stretch's own from its first slot's number on
};

TablePlan plan_table(void *workspace, int64_t m, int partitions, size_t *bytes) {
  TablePlan tp{};
  tp.per_part = m / partitions;
  const int64_t most = kMaxStretches / partitions > 0 ? kMaxStretches / partitions : 1;
  tp.len = ceil_div(ceil_div(tp.per_part > 0 ? tp.per_part : 1, most), kStep) * kStep;
  tp.cpp = ceil_div(tp.per_part, tp.len);
  tp.count = tp.cpp * partitions;
  Carver cv(workspace);
  tp.found = cv.take<uint32_t>((size_t)tp.count);
  tp.at = cv.take<uint32_t>((size_t)tp.count + 1);
  tp.entries = cv.take<int32_t>((size_t)(tp.per_part * partitions));
  *bytes = cv.used;
  return tp;
}

__device__ inline bool filled(int32_t e) { return (e & 0x7fffffff) != 0; }

// Zeroed words in which finished workgroups count themselves and their entries: per group of up to kMarkGroup
// workgroups of a partition, then per partition, then once per partition in `done`.  (Adds to one word are carried out
// one after the other, 11 ns each.)
struct TableMarks {
  unsigned long long *group;
  unsigned long long *part;
  uint32_t *done;
  uint32_t parts, per_part, groups;  // partitions; workgroups and groups of one
};
constexpr int kMarkShift = 40;  // arrivals above, entries below

// The entries of stretch w (of partition `part`) to the workspace: how many there are; `bad` if one is no index.
__device__ inline uint32_t walk_stretch(const int32_t *__restrict__ table, int64_t n, const TablePlan &tp, int64_t part,
                                        int64_t w, bool &bad) {
  const int64_t lo = part * tp.per_part + (w - part * tp.cpp) * tp.len;
  const int64_t last = (part + 1) * tp.per_part;
  const int64_t hi = lo + tp.len < last ? lo + tp.len : last;
  const int lane = lane_id();
  // vectors start at multiples of 16 bytes in memory, whatever the table's address and the partition's edge are
  const int64_t off = (int64_t)((reinterpret_cast<uintptr_t>(table) >> 2) & 3u);
  const int64_t first = ((lo + off) & ~(int64_t)3) - off;  // at most three slots in front of the stretch
  auto load = [&](int64_t base, int4 (&q)[kRows]) {
    if (base >= lo && base + kStep <= hi) {
#pragma unroll
      for (int r = 0; r < kRows; ++r) q[r] = *reinterpret_cast<const int4 *>(table + base + r * kRow + lane * 4);
    } else {
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        const int64_t s = base + r * kRow + lane * 4;
        q[r].x = s >= lo && s < hi ? table[s] : 0;
        q[r].y = s + 1 >= lo && s + 1 < hi ? table[s + 1] : 0;
        q[r].z = s + 2 >= lo && s + 2 < hi ? table[s + 2] : 0;
        q[r].w = s + 3 >= lo && s + 3 < hi ? table[s + 3] : 0;
      }
    }
  };
  int32_t *out = tp.entries + lo;
  uint32_t found = 0;
  int4 q[kRows], next[kRows];
  load(first, next);
#pragma unroll 1
  for (int64_t base = first; base < hi; base += kStep) {
#pragma unroll
    for (int r = 0; r < kRows; ++r) q[r] = next[r];
    if (base + kStep < hi) load(base + kStep, next);  // on its way while these rows are looked at
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int32_t e[4] = {q[r].x, q[r].y, q[r].z, q[r].w};
      uint32_t c = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) c += filled(e[j]) ? 1u : 0u;
      const uint32_t incl = wave_inclusive_scan(c);
      uint32_t pos = found + incl - c;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (filled(e[j])) {
          out[pos++] = e[j];
          bad |= (int64_t)e[j] + n < 0 || (int64_t)e[j] >= n;
        }
      }
      found += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    }
  }
  return found;
}

template <bool MARKED>
__global__ __launch_bounds__(kBlock, 8) void k_table_walk(const int32_t *__restrict__ table, int64_t n, TablePlan tp,
                                                          TableMarks marks, int64_t *__restrict__ splits,
                                                          HostAnswer answer, int32_t *status) {
  constexpr int kWaves = kBlock / 64;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int64_t part, w;
  if (MARKED) {  // a workgroup's stretches are of one partition
    part = blockIdx.x / marks.per_part;
    w = (int64_t)(blockIdx.x - (uint32_t)part * marks.per_part) * kWaves + wave;
    w = w < tp.cpp ? part * tp.cpp + w : tp.count;
  } else {
    w = (int64_t)blockIdx.x * kWaves + wave;
    part = w / tp.cpp;
  }
  uint32_t found = 0;
  if (w < tp.count) {
    bool bad = false;
    found = walk_stretch(table, n, tp, part, w, bad);
    const uint64_t any_bad = __ballot(bad);
    if (lane_id() == 0) {
      tp.found[w] = found;
      if (any_bad) atomicOr(status, ZEN_STAT_BAD_INDEX);
    }
  }
  if (!MARKED) return;
  __shared__ uint32_t held[kWaves];
  __shared__ bool last;
  if (lane_id() == 0) {
    held[wave] = found;
    wait_global_acks();  // the wave's share of the status word
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    constexpr unsigned long long kEntries = (1ull << kMarkShift) - 1ull, kArrived = 1ull << kMarkShift;
    unsigned long long mine = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) mine += held[i];
    const uint32_t own = blockIdx.x - (uint32_t)part * marks.per_part;
    const uint32_t group = own / kMarkGroup;
    const uint32_t left = marks.per_part - group * kMarkGroup;
    last = false;
    unsigned long long old = atomicAdd(&marks.group[(uint32_t)part * marks.groups + group], kArrived | mine);
    if ((old >> kMarkShift) + 1u == (left < (uint32_t)kMarkGroup ? left : (uint32_t)kMarkGroup)) {
      mine += old & kEntries;
      old = atomicAdd(&marks.part[part], kArrived | mine);
      if ((old >> kMarkShift) + 1u == marks.groups) last = atomicAdd(marks.done, 1u) == marks.parts - 1u;
    }
  }
  __syncthreads();
  if (!last) return;
  for (uint32_t p = threadIdx.x; p < marks.parts; p += kBlock) {
    const int64_t size = (int64_t)(__hip_atomic_load(&marks.part[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &
                                   ((1ull << kMarkShift) - 1ull));
    splits[p] = size;
    host_store(answer.host + 1 + p, size);
  }
  if (threadIdx.x == 0)
    host_store(answer.host + 1 + marks.parts, (int64_t)__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  host_answered(answer);
}

// Places of the stretches and the partitions' sizes.  One workgroup, one round: there are 8192 stretches unless there
// are more partitions than that.
__global__ __launch_bounds__(kScanBlock) void k_table_offsets(TablePlan tp, int partitions,
                                                              int64_t *__restrict__ splits) {
  constexpr int kEach = 8;
  __shared__ uint32_t smem[kScanBlock / 64 + 1];
  uint32_t before = 0;
  for (int64_t c0 = 0; c0 < tp.count; c0 += kScanBlock * kEach) {
    const int64_t first = c0 + (int64_t)threadIdx.x * kEach;
    uint32_t v[kEach], sum = 0;
#pragma unroll
    for (int j = 0; j < kEach; ++j) v[j] = first + j < tp.count ? tp.found[first + j] : 0u;
#pragma unroll
    for (int j = 0; j < kEach; ++j) sum += v[j];
    uint32_t total;
    uint32_t at = before + block_exclusive_scan<uint32_t, kScanBlock>(sum, smem, &total);
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      if (first + j < tp.count) tp.at[first + j] = at;
      at += v[j];
    }
    before += total;
  }
  if (threadIdx.x == 0) tp.at[tp.count] = before;
  __syncthreads();
  for (int64_t p = threadIdx.x; p < partitions; p += kScanBlock)
    splits[p] = (int64_t)tp.at[(p + 1) * tp.cpp] - (int64_t)tp.at[p * tp.cpp];
}

// PLACED: k_table_offsets has left the stretches' places; else they are sums of the counts in front of them.
template <typename S, bool PLACED>
__global__ __launch_bounds__(kMoveBlock) void k_table_gather(const S *__restrict__ in, int64_t n, TablePlan tp,
                                                             int32_t *__restrict__ out_idx, S *__restrict__ out_val,
                                                             int64_t total) {
  constexpr int kWaves = kMoveBlock / 64;
  static_assert(kWaves == 4, "a workgroup's counts are a vector");
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t w = (int64_t)blockIdx.x * kWaves + wave;
  uint32_t at = 0;
  if (!PLACED) {
    __shared__ uint32_t sums[kWaves];
    const uint4 *found = reinterpret_cast<const uint4 *>(tp.found);
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kMoveBlock) {
      const uint4 q = found[i];
      sum += (q.x + q.y) + (q.z + q.w);
    }
    sum = wave_sum(sum);
    if (lane_id() == 0) sums[wave] = sum;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) at += sums[i];
    for (int i = 0; i < wave; ++i) at += w < tp.count ? tp.found[(int64_t)blockIdx.x * kWaves + i] : 0u;
    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
  }
  if (w >= tp.count) return;
  if (PLACED) at = tp.at[w];
  const int64_t part = w / tp.cpp;
  const int32_t *from = tp.entries + part * tp.per_part + (w - part * tp.cpp) * tp.len;
  const uint32_t mine = tp.found[w];
  constexpr uint32_t kAhead = 4;
  for (uint32_t i0 = 0; i0 < mine; i0 += 64 * kAhead) {
    int32_t k[kAhead];
    S v[kAhead];
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j) {
      const uint32_t i = i0 + j * 64 + (uint32_t)lane_id();
      k[j] = from[i < mine ? i : 0u];
    }
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j) {
      const int64_t t = k[j] < 0 ? (int64_t)k[j] + n : (int64_t)k[j];  // a negative index counts from the end
      v[j] = t >= 0 && t < n ? in[t] : S(0);
    }
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j) {
      const uint32_t i = i0 + j * 64 + (uint32_t)lane_id();
      if (i < mine && (int64_t)at + i < total) {
        out_idx[at + i] = k[j];
        out_val[at + i] = v[j];
      }
    }
  }
}

int table_find(const int32_t *table, int64_t n, const TablePlan &tp, int partitions, int64_t *splits, int32_t *status,
               hipStream_t s) {
  k_table_walk<false><<<dim3((unsigned)ceil_div(tp.count, kBlock / 64)), dim3(kBlock), 0, s>>>(
      table, n, tp, TableMarks{}, nullptr, HostAnswer{}, status);
  ZEN_LAUNCH_CHECK("k_table_walk");
  k_table_offsets<<<dim3(1), dim3(kScanBlock), 0, s>>>(tp, partitions, splits);
  ZEN_LAUNCH_CHECK("k_table_offsets");
  return ZEN_OK;
}

template <typename S>
int table_gather(const void *input, int64_t n, const TablePlan &tp, int partitions, int32_t *out_idx, void *out_val,
                 int64_t total, hipStream_t s) {
  const auto kernel = partitions > kMostMarked ? k_table_gather<S, true> : k_table_gather<S, false>;
  kernel<<<dim3((unsigned)ceil_div(tp.count, kMoveBlock / 64)), dim3(kMoveBlock), 0, s>>>(
      static_cast<const S *>(input), n, tp, out_idx, static_cast<S *>(out_val), total);
  ZEN_LAUNCH_CHECK("k_table_gather");
  return ZEN_OK;
}

int table_args(const char *what, const int32_t *table, int64_t m, int partitions, int64_t n, void *workspace,
               size_t workspace_bytes) {
  if (partitions < 1 || m < partitions || m > 0x7fffffffll || n < 0 || n > 0x7fffffffll || !table || !workspace)
    return fail(ZEN_EINVAL, what);
  if (workspace_bytes < zen_table_lists_workspace(m, partitions)) return fail(ZEN_EWORKSPACE, what);
  return ZEN_OK;
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_table_lists_workspace(int64_t m, int partitions) {
  if (partitions < 1 || m < 0) return 0;
  size_t bytes;
  (void)zen::plan_table(nullptr, m, partitions, &bytes);
  return bytes;
}

int zen_table_find(const int32_t *table, int64_t m, int partitions, int64_t n, int64_t *splits, void *workspace,
                   size_t workspace_bytes, int32_t *status, void *stream) {
  using namespace zen;
  if (!splits || !status) return fail(ZEN_EINVAL, "zen_table_find: null pointer");
  const int rc = table_args("zen_table_find: bad argument or workspace", table, m, partitions, n, workspace,
                            workspace_bytes);
  if (rc != ZEN_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  size_t bytes;
  const TablePlan tp = plan_table(workspace, m, partitions, &bytes);
  return table_find(table, n, tp, partitions, splits, status, s);
}

int zen_table_find_sizes(const int32_t *table, int64_t m, int partitions, int64_t n, int64_t *splits, int64_t *marks,
                         void *workspace, size_t workspace_bytes, int32_t *status, int64_t *host, int64_t words,
                         void *stream) {
  using namespace zen;
  if (!splits || !marks || !status) return fail(ZEN_EINVAL, "zen_table_find_sizes: null pointer");
  if (partitions > kMostMarked) return fail(ZEN_EINVAL, "zen_table_find_sizes: too many partitions");
  int rc = table_args("zen_table_find_sizes: bad argument or workspace", table, m, partitions, n, workspace,
                      workspace_bytes);
  if (rc != ZEN_OK) return rc;
  HostAnswer answer;
  rc = host_ask(host, words, (int64_t)partitions + 1, &answer);
  if (rc != ZEN_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  size_t bytes;
  const TablePlan tp = plan_table(workspace, m, partitions, &bytes);
  TableMarks tm;
  tm.parts = (uint32_t)partitions;
  tm.per_part = (uint32_t)ceil_div(tp.cpp, (int64_t)(kBlock / 64));
  tm.groups = (uint32_t)ceil_div((int64_t)tm.per_part, (int64_t)kMarkGroup);
  tm.group = reinterpret_cast<unsigned long long *>(marks);
  tm.part = tm.group + (size_t)tm.groups * tm.parts;
  tm.done = reinterpret_cast<uint32_t *>(tm.part + tm.parts);
  k_table_walk<true><<<dim3(tm.per_part * tm.parts), dim3(kBlock), 0, s>>>(table, n, tp, tm, splits, answer, status);
  const hipError_t e = hipGetLastError();
  return host_finish(e == hipSuccess ? ZEN_OK : hip_fail(e, "k_table_walk"), answer, s);
}

int zen_table_gather(const int32_t *table, int64_t m, int partitions, const void *input, int dtype, int64_t n,
                     int32_t *out_idx, void *out_val, int64_t total, void *workspace, size_t workspace_bytes,
                     void *stream) {
  using namespace zen;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_table_gather: bad dtype");
  const int rc = table_args("zen_table_gather: bad argument or workspace", table, m, partitions, n, workspace,
                            workspace_bytes);
  if (rc != ZEN_OK) return rc;
  if (total <= 0) return ZEN_OK;
  if (!out_idx || !out_val || !input) return fail(ZEN_EINVAL, "zen_table_gather: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  size_t bytes;
  const TablePlan tp = plan_table(workspace, m, partitions, &bytes);
  return dtype == ZEN_BF16 ? table_gather<uint16_t>(input, n, tp, partitions, out_idx, out_val, total, s)
                           : table_gather<uint32_t>(input, n, tp, partitions, out_idx, out_val, total, s);
}

}  // extern "C"
