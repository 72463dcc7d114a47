// Shared host/device helpers for libzen_hip (gfx950, wave64 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "zen_hip.h"

namespace zen {

// ------------------------------------------------------------------ host side

extern thread_local char g_last_error[256];

inline int fail(int code, const char *what) {
  snprintf(g_last_error, sizeof(g_last_error), "%s", what);
  return code;
}

inline int hip_fail(hipError_t e, const char *where) {
  snprintf(g_last_error, sizeof(g_last_error), "%s: %s", where, hipGetErrorString(e));
  return ZEN_EHIP;
}

#define ZEN_HIP_CHECK(expr)                                      \
  do {                                                           \
    hipError_t zen_e_ = (expr);                                  \
    if (zen_e_ != hipSuccess) return ::zen::hip_fail(zen_e_, #expr); \
  } while (0)

#define ZEN_LAUNCH_CHECK(name)                                   \
  do {                                                           \
    hipError_t zen_e_ = hipGetLastError();                       \
    if (zen_e_ != hipSuccess) return ::zen::hip_fail(zen_e_, name); \
  } while (0)

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Carves 256-byte aligned sub-buffers out of one workspace.
struct Carver {
  char *base;
  size_t used = 0;
  explicit Carver(void *p) : base(static_cast<char *>(p)) {}
  template <typename T>
  T *take(size_t count) {
    T *p = reinterpret_cast<T *>(base + used);
    used += align_up(count * sizeof(T), 256);
    return p;
  }
};

inline int ceil_log2_u64(uint64_t x) {  // bits needed to represent values in [0, x]
  int b = 0;
  while (b < 64 && (x >> b) != 0) ++b;
  return b;
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Kernel timing tags (zen_profile.hip).  A ProfScope around a launch records
// HIP events on the launch stream when profiling is enabled; otherwise it is
// one relaxed load of a flag and a branch.
enum ProfTag {
  kProfTopkHist = 0,
  kProfSelectCompact,
  kProfInsertList,
  kProfFinalKey,
  kProfSort,
  kProfGather,
  kProfMergePrep,
  kProfMergeReduce,
  kProfCompress,
  kProfInsertDense,
  kProfSelectStage,
  kProfFeed,
  kProfSlabSort,
  kProfSlabChains,
  kProfSlabPlace,
  kProfMergeFeed,
  kProfMergeBucket,
  kProfSampleHist,
  kProfDecodeFused,
  kProfWideTail,
  kProfWideScatter,
  kProfWideMerge,
  kProfCount
};

class ProfScope {
 public:
  ProfScope(int tag, hipStream_t stream);
  ~ProfScope();
  ProfScope(const ProfScope &) = delete;
  ProfScope &operator=(const ProfScope &) = delete;

 private:
  int tag_;
  hipStream_t stream_;
  hipEvent_t start_, stop_;
};

// ---------------------------------------------------------------- device side

constexpr uint32_t kSeed1 = 10001861u;  // functions_cuda_kernel.cu:101
constexpr uint32_t kSeed2 = 100703u;    // functions_cuda_kernel.cu:124
constexpr uint32_t kSeed3 = 5002639u;   // functions_cuda_kernel.cu:151

// functions_cuda_kernel.cu:80-88 without the additive seed, in Horner form
// (identical in uint32 ring arithmetic).  h(k, c) = poly(k) + c.
__host__ __device__ inline uint32_t poly(uint32_t k) {
  return ((573729859u * k + 0xcc9e2d51u) * k + 0x1b873593u) * k;
}

// Probe geometry of the hash table: level 0 probes the whole table, levels 1
// and 2 probe inside the partition level 0 landed in
// (functions_cuda_kernel.cu:101-107, 119-129, 144-156).
struct Probe {
  uint32_t m;    // table size
  uint32_t npp;  // slots per partition = m / partitions
  int levels;    // 1, 2 or 3
};

__device__ inline uint32_t probe_slot(const Probe &g, uint32_t t, int level, uint32_t *part_out) {
  const uint32_t h = poly(t);
  const uint32_t first = (h + kSeed1) % g.m;
  const uint32_t part = first / g.npp;
  *part_out = part;
  if (level == 0) return first;
  const uint32_t seed = level == 1 ? kSeed2 : kSeed3;
  return part * g.npp + (h + seed) % g.npp;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Element storage and magnitude keys (bit pattern with the sign cleared).
template <typename S>
struct KeyOf;
template <>
struct KeyOf<uint16_t> {
  static constexpr uint32_t kMask = 0x7fffu;
  static constexpr int kBits = 15;
  static __device__ inline float to_f32(uint16_t v) { return __uint_as_float(uint32_t(v) << 16); }
};
template <>
struct KeyOf<uint32_t> {
  static constexpr uint32_t kMask = 0x7fffffffu;
  static constexpr int kBits = 31;
  static __device__ inline float to_f32(uint32_t v) { return __uint_as_float(v); }
};

__device__ inline uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x0040u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

// What a merge writes for a sum: the fp32 sum itself, or the sum rounded once to bf16 (a sum that rounds to zero is
// dropped with those that are zero; torch.nonzero keeps NaN and drops +-0).
template <typename O>
struct SumAs;
template <>
struct SumAs<float> {
  static __device__ inline float of(float v) { return v; }
  static __device__ inline bool kept(float v) { return v != 0.0f; }
};
template <>
struct SumAs<uint16_t> {
  static __device__ inline uint16_t of(float v) { return f32_to_bf16_rne(v); }
  // (half of the smallest bf16 rounds to even, that is to zero; NaN is kept)
  static __device__ inline bool kept(float v) { return (__float_as_uint(v) & 0x7fffffffu) > 0x8000u; }
};

// Waits until the global memory operations this wave has issued, stores and atomics without a return value
// included, have been acknowledged by the place that carries them out.
__device__ inline void wait_global_acks() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Reads a word that other workgroups of the running kernel have changed with device-wide atomics, from the
// place where those are carried out (not from this compute unit's caches).
__device__ inline uint32_t load_fresh(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Counts workgroup `index` of `total` as finished (by one thread of it, once what the last one is to find has been carried
// out); true for the last of them.  A word takes one add after the other, ten nanoseconds each, and workgroups that end
// together would stand in line for it: they count in kDoneGroups words, and the last of each group in one more (the select
// kernel's 768 workgroups on 62 M bf16 elements 35.2 us with one word, 31.8 so; 1536 of k_merge_bucket 87.8 and 79.4).
// words: kDoneWords of them, zero, each counter in a memory line of its own.
constexpr uint32_t kDoneGroups = 16, kDonePad = 32;
constexpr uint32_t kDoneWords = (kDoneGroups + 1) * kDonePad;
__device__ inline bool done_last(uint32_t *words, uint32_t index, uint32_t total) {
  const uint32_t g = index % kDoneGroups, groups = total < kDoneGroups ? total : kDoneGroups;
  if (atomicAdd(&words[g * kDonePad], 1u) != (total - g + kDoneGroups - 1u) / kDoneGroups - 1u) return false;
  return atomicAdd(&words[kDoneGroups * kDonePad], 1u) == groups - 1u;
}

// Ascending compare-exchange network (bitonic with mirrored first step), valid for any n: positions >= n act as
// +infinity and never move.  By the whole workgroup.
template <typename T>
__device__ inline void sort_network(T *a, uint32_t n) {
  uint32_t steps = 0;
  while ((1u << steps) < n) ++steps;
  const uint32_t half = (1u << steps) >> 1;
  auto exchange = [&](uint32_t i, uint32_t l) {
    if (l >= n) return;
    const T x = a[i], y = a[l];
    if (x > y) {
      a[i] = y;
      a[l] = x;
    }
  };
  for (uint32_t k = 0; k < steps; ++k) {  // sorted runs of 2^k become runs of 2^(k + 1)
    for (uint32_t q = threadIdx.x; q < half; q += blockDim.x) {
      const uint32_t first = q >> k << (k + 1), r = q & ((1u << k) - 1u);
      exchange(first + r, first + (2u << k) - 1u - r);
    }
    __syncthreads();
    for (uint32_t j = k; j-- > 0;) {
      for (uint32_t q = threadIdx.x; q < half; q += blockDim.x) {
        const uint32_t i = (q >> j << (j + 1)) + (q & ((1u << j) - 1u));
        exchange(i, i + (1u << j));
      }
      __syncthreads();
    }
  }
}

// Where the host waits for what a call has to know there (zen_readback.hip): pinned words, of which word 0 takes the
// ticket once the others hold the answer.  The kernel that knows the answer stores it, where that is one of the call's
// own: no launch for it, and what is left of the call's work runs while the host goes on.
struct HostAnswer {
  int64_t *host = nullptr;  // null: nobody asks
  int64_t ticket = 0;
};
struct HostAsk {  // the same on its way through host code
  HostAnswer answer;
  bool *answered = nullptr;  // set where kernels of the call's own answer
};
// Past the caches, so that nothing has to be written back for the host to see it.
__device__ inline void host_store(int64_t *p, int64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// By the whole workgroup, behind its stores of the answer's words.
__device__ inline void host_answered(const HostAnswer &a) {
  wait_global_acks();
  __syncthreads();
  if (threadIdx.x == 0) host_store(a.host, a.ticket);
}
// A count and the status word behind it (no count: the status word alone), once every workgroup that changes them has
// been waited for.  By the whole workgroup.
__device__ inline void host_answer_count(const HostAnswer &a, const int64_t *count, const int32_t *status) {
  if (!a.host) return;
  if (threadIdx.x == 0) {
    if (count) host_store(a.host + 1, __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    host_store(a.host + (count ? 2 : 1), (int64_t)__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  host_answered(a);
}

__device__ inline int lane_id() { return int(__lane_id()); }

__device__ inline uint64_t lanes_below() {  // mask of lanes with a smaller id
  return (1ull << lane_id()) - 1ull;
}

// Inclusive prefix sum across the 64 lanes: DPP row shifts and broadcasts, six additions.  (Through LDS permutes every
// step waits for a round trip: an all-reduce of a 62 M-element bucket, 10 % selected: 622 us of kernels, now 607.)
__device__ inline uint32_t wave_inclusive_scan(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1,3
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2,3
  return x;
}
__device__ inline uint64_t wave_inclusive_scan(uint64_t x) {
  // one DPP step on both halves; what moves in is 0 where the mask leaves a row out
#define ZEN_STEP(ctrl, rows)                                                                                             \
  {                                                                                                                      \
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, ctrl, rows, 0xf, false);              \
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), ctrl, rows, 0xf, false);      \
    x += ((uint64_t)hi << 32) | lo;                                                                                      \
  }
  ZEN_STEP(0x111, 0xf)
  ZEN_STEP(0x112, 0xf)
  ZEN_STEP(0x114, 0xf)
  ZEN_STEP(0x118, 0xf)
  ZEN_STEP(0x142, 0xa)
  ZEN_STEP(0x143, 0xc)
#undef ZEN_STEP
  return x;
}

// Sum over the 64 lanes (all of them active), in every lane.
__device__ inline uint32_t wave_sum(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive_scan(v), 63);
}
__device__ inline uint64_t wave_sum(uint64_t v) {
  const uint64_t s = wave_inclusive_scan(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)s, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(s >> 32), 63);
  return ((uint64_t)hi << 32) | lo;
}

// The value lane `lane` (the same for the whole wave) holds.
__device__ inline uint32_t wave_read(uint32_t v, int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lane); }
__device__ inline uint64_t wave_read(uint64_t v, int lane) {
  return ((uint64_t)wave_read((uint32_t)(v >> 32), lane) << 32) | wave_read((uint32_t)v, lane);
}

// The inclusive scan's steps inside rows of sixteen lanes.
__device__ inline uint32_t row_inclusive_scan(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
  return x;
}
__device__ inline uint64_t row_inclusive_scan(uint64_t x) {
#define ZEN_STEP(ctrl)                                                                                                   \
  {                                                                                                                      \
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, ctrl, 0xf, 0xf, false);               \
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), ctrl, 0xf, 0xf, false);       \
    x += ((uint64_t)hi << 32) | lo;                                                                                      \
  }
  ZEN_STEP(0x111)
  ZEN_STEP(0x112)
  ZEN_STEP(0x114)
  ZEN_STEP(0x118)
#undef ZEN_STEP
  return x;
}

// Exclusive scan over the threads of a block (all of them active).  `total` receives the block sum in every thread.
// smem needs BLOCK/64 + 1 T's.  The waves' sums are scanned by the lanes of every wave, a lane a sum (a row of sixteen
// lanes holds them all): the kernels of a thousand threads that scan between their steps are bound by vector instructions
// and by the chain of their phases, and a loop over sixteen sums in every thread is 64 instructions (k_slab_sort of 3.1 M
// bf16 records 17.9 us, 17.0 so; k_wide_merge of as many 39.9 and 38.0).
template <typename T, int BLOCK>
__device__ inline T block_exclusive_scan(T v, T *smem, T *total) {
  constexpr int kWaves = BLOCK / 64;
  static_assert(BLOCK % 64 == 0 && kWaves >= 1 && kWaves <= 16 && (kWaves & (kWaves - 1)) == 0, "a row of lanes holds the waves' sums");
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const T incl = wave_inclusive_scan(v);
  if (lane_id() == 63) smem[wave] = incl;
  __syncthreads();
  const T own = smem[lane_id() & (kWaves - 1)];
  const T upto = row_inclusive_scan(own);  // right in the first kWaves lanes
  __syncthreads();
  *total = wave_read(upto, kWaves - 1);
  return wave_read(upto - own, wave) + incl - v;
}

// ------------------------------------------------ single-pass prefix over tiles
// Decoupled look-back.  One 64-bit descriptor per tile holds 2 flag bits and a
// 62-bit value, so flag and value are published by one atomic store: first the
// tile's own count (aggregate), later its inclusive prefix.  A tile sums the
// aggregates of its predecessors, 64 at a time, back to the nearest one that
// already shows a prefix.  Tiles take their id from a ticket counter, so every
// lower-numbered tile already runs and the wait cannot deadlock; it is also
// bounded.  The prefix frontier advances 64 tiles per memory round trip, so
// kernels keep their tile count in the low thousands.
//
// Scratch layout (all zero before the launch): ntiles descriptors and one
// ticket word = scan_words(ntiles) uint64.

constexpr uint64_t kDescAggregate = 1ull << 62;
constexpr uint64_t kDescPrefix = 2ull << 62;
constexpr uint64_t kDescValue = (1ull << 62) - 1;
constexpr uint32_t kSpinLimit = 1u << 22;  // bounded wait: flag ZEN_STAT_INTERNAL instead of hanging

constexpr size_t scan_words_c(int64_t ntiles) { return (size_t)ntiles + 2; }
inline size_t scan_words(int64_t ntiles) { return scan_words_c(ntiles); }

struct ScanState {
  unsigned long long *desc;
  uint32_t *ticket;
};

inline ScanState scan_state(void *scratch, int64_t ntiles) {
  ScanState st;
  st.desc = static_cast<unsigned long long *>(scratch);
  st.ticket = reinterpret_cast<uint32_t *>(st.desc + ntiles);
  return st;
}

__device__ inline uint64_t desc_load(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void desc_store(unsigned long long *p, uint64_t v) {
  __hip_atomic_store(p, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Called by every thread of the block.  Returns the sum of the aggregates of
// all tiles before `tile`.  smem: one uint64.
__device__ inline uint64_t lookback_exclusive(const ScanState &st, int tile, uint64_t aggregate,
                                              int32_t *status, uint64_t *smem) {
  unsigned long long *desc = st.desc;
  if (threadIdx.x < 64) {
    const int lane = lane_id();
    if (lane == 0) desc_store(&desc[tile], (tile == 0 ? kDescPrefix : kDescAggregate) | aggregate);
    uint64_t excl = 0;
    if (tile > 0) {
      int base = tile - 1;
      bool gave_up = false;
      for (;;) {
        const int p = base - lane;
        uint64_t d = kDescPrefix;  // tiles before the first: prefix 0
        if (p >= 0) {
          d = desc_load(&desc[p]);
          uint32_t spins = 0;
          while ((d >> 62) == 0) {
            if (++spins > kSpinLimit) {
              gave_up = true;
              d = kDescPrefix;
              break;
            }
            __builtin_amdgcn_s_sleep(2);
            d = desc_load(&desc[p]);
          }
        }
        const uint64_t have_prefix = __ballot((d >> 62) == 2);
        const int first = have_prefix ? __ffsll((unsigned long long)have_prefix) - 1 : 64;
        excl += wave_sum(lane <= first ? (uint64_t)(d & kDescValue) : (uint64_t)0);
        if (have_prefix) break;
        base -= 64;
      }
      if (gave_up) atomicOr(status, ZEN_STAT_INTERNAL);
      if (lane == 0) desc_store(&desc[tile], kDescPrefix | (excl + aggregate));
    }
    if (lane == 0) *smem = excl;
  }
  __syncthreads();
  const uint64_t r = *smem;
  __syncthreads();
  return r;
}

// Grid-stride fill; also the way to clear scratch without a memset node.
template <typename T>
__global__ void k_fill(T *p, T v, size_t count) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

template <typename T>
inline void launch_fill(T *p, T v, size_t count, hipStream_t s) {
  if (count == 0) return;
  const size_t blocks = (count + 1023) / 1024;
  k_fill<T><<<dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, s>>>(p, v, count);
}

// ---------------------------------------------------------- sort (zen_sort.hip)

// Stable LSD radix sort of (key, val) pairs on the low `bits` bits.  The result
// ends in (keys_a, vals_a) when the returned value is 0 and in (keys_b,
// vals_b) when it is 1; negative = error.  `scratch` from sort_scratch_bytes.
// more_a / more_b: an optional second payload moved along with the first.
size_t sort_scratch_bytes(int64_t max_count);
int sort_pairs(uint32_t *keys_a, uint32_t *vals_a, uint32_t *keys_b, uint32_t *vals_b,
               int64_t max_count, const uint32_t *count_dev, int bits, void *scratch,
               int32_t *status, hipStream_t stream, uint32_t *more_a = nullptr, uint32_t *more_b = nullptr);

// Stable sort of records whose keys spread evenly over [0, sentinel) (hash slots, hashed indices): one
// scatter pass into 511 key ranges, then each range sorted inside LDS by one workgroup.  Records with
// key >= sentinel come last, in no particular order.  The result is in the b arrays (returns 1; negative =
// error).  A key range holding more records than fit in LDS sets ZEN_STAT_RETRY in *status and the order
// is then unspecified.  bucket_sort_fits: whether `expected` records (the live count may sit on the device)
// leave the key ranges room to spare; same scratch as sort_pairs.
bool bucket_sort_fits(int64_t expected, uint32_t sentinel);
int bucket_sort_pairs(uint32_t *keys_a, uint32_t *vals_a, uint32_t *keys_b, uint32_t *vals_b, int64_t max_count,
                      const uint32_t *count_dev, uint32_t sentinel, void *scratch, int32_t *status,
                      hipStream_t stream, uint32_t *more_a = nullptr, uint32_t *more_b = nullptr);

// ------------------------------------------------- answers to the host (zen_readback.hip)

// The answer a call on `host` (words of them) with `need` words besides word 0 will get; null words: an error.
int host_ask(int64_t *host, int64_t words, int64_t need, HostAnswer *answer);
// One kernel that answers with the words two arrays hold, for calls whose kernels do not.
int host_answer_launch(const HostAnswer &answer, const int64_t *first, int n0, const int32_t *second, int n1, hipStream_t s);
// The end of a call that asked, `rc` of its launches: returns when the answer is there, or with an error (the stream's
// among them) when no answer to this call can come any more.
int host_finish(int rc, const HostAnswer &answer, hipStream_t s);

}  // namespace zen
