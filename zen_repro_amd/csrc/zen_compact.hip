// Ordered compaction of a dense tensor: ascending indices and values of the selected elements (zen_select;
// encode_sparse_tensor, comm.py:47-50).
//
// The tensor is cut into one stretch per wave.  A wave walks its stretch on its own, with no barrier and nobody to
// wait for, and leaves what it selects side by side in a part of the workspace that is its own (k_compact_walk);
// a second kernel sums up the counts in front of every stretch and moves the entries to their places
// (k_compact_move).  A stretch with more than an eighth of its elements selected does not fit its part: the second
// kernel walks it again and writes it straight to its place.  Up to kOneMax elements one workgroup does both steps
// in one launch.
// Bound by the read of the tensor and the extraction of what is selected (62 M bf16 elements, 4.4 % selected: 28 + 12
// us, of which the read alone would take 18).  A single pass with tiles chained by
// look-back took 88 us there: thousands of tiles draw their numbers from one counter, 11 ns each, and wait for
// each other's prefixes.
#include "zen_select.h"

namespace zen {
namespace {

constexpr int kBlock = 256;                 // of the walking kernel
constexpr int kMoveBlock = 1024;            // of the moving kernel: a stretch per wave
constexpr int kMoveWaves = kMoveBlock / 64;
constexpr int kRows = 4;                    // rows of one 16-byte vector per lane in flight
constexpr int64_t kMaxStretches = 8192;     // 32 waves per compute unit
constexpr int64_t kOneMax = 65536;
template <typename S>
constexpr int row() { return 64 * VecOf<S>::kN; }  // elements of a row
template <typename S>
constexpr int64_t least_stretch() { return (int64_t)row<S>() * kRows; }

// Flags of the elements of one vector, element e at bit e.
__device__ inline uint32_t vec_flags(const uint4 &q, uint32_t least, uint16_t) {
  const uint32_t c = (0x8000u - least) * 0x00010001u;  // per 16-bit half: key + c carries into bit 15 iff key >= least
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
  uint32_t x = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t m = ((w[j] & 0x7fff7fffu) + c) & 0x80008000u;
    x |= (((m >> 15) | (m >> 30)) & 3u) << (2 * j);
  }
  return x;
}
__device__ inline uint32_t vec_flags(const uint4 &q, uint32_t least, uint32_t) {
  return ((q.x & 0x7fffffffu) >= least ? 1u : 0u) | ((q.y & 0x7fffffffu) >= least ? 2u : 0u) |
         ((q.z & 0x7fffffffu) >= least ? 4u : 0u) | ((q.w & 0x7fffffffu) >= least ? 8u : 0u);
}
__device__ inline uint16_t vec_pick(const uint4 &q, uint32_t e, uint16_t) {
  const uint32_t a = e & 2u ? q.y : q.x, b = e & 2u ? q.w : q.z;
  const uint32_t w = e & 4u ? b : a;
  return (uint16_t)(e & 1u ? w >> 16 : w);
}
__device__ inline uint32_t vec_pick(const uint4 &q, uint32_t e, uint32_t) {
  const uint32_t a = e & 1u ? q.y : q.x, b = e & 1u ? q.w : q.z;
  return e & 2u ? b : a;
}

// Sixteen bytes from an address that is a multiple of 16 or, !ALIGNED, of an element's size only (a view that begins
// at an odd element): one load either way.  ONCE: nobody looks at them again (a streamed load).
template <typename S, bool ALIGNED, bool ONCE>
__device__ inline uint4 load16(const S *at) {
  uint4 q;
  if (ALIGNED && ONCE) {
    const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(at));
    __builtin_memcpy(&q, &t, 16);
  } else if (ALIGNED) {
    q = *reinterpret_cast<const uint4 *>(at);
  } else {
    __builtin_memcpy(&q, at, 16);
  }
  return q;
}

// What a wave has found and not yet written out.  A store on its way holds up the next rows' elements (a wave's loads
// are waited for together with the stores behind them), so that the walk keeps its findings here and writes them out
// together: 62 M bf16 elements, 3.4 % found, 32 us with each written at once, 27.6 so (and the move behind it 11.1 and
// 8.8, since a streamed tensor leaves the findings in the caches); 62 M fp32 elements, 10 % found, 67 and 56.  The
// read alone takes 21.
constexpr uint32_t kHeld = 512;
template <typename S>
struct Held {
  int32_t idx[kHeld];
  S val[kHeld];
};

// A wave's walk over elements [begin, end) (begin a multiple of the vector length): selected element number i goes
// to idx[i], val[i] if i < room.  Returns how many there are.  WRITE == false: only counts.  A stretch holds fewer
// than 2^18 elements, so that byte offsets from the (uniform) pointers fit 32 bits.  HOLD: by way of `held`.
template <typename S, bool ALIGNED, bool WRITE, bool HOLD = false, typename I>
__device__ __forceinline__ uint32_t walk(const S *__restrict__ in, int64_t begin, int64_t end, uint32_t least,
                                I *__restrict__ idx, S *__restrict__ val, uint32_t room, Held<S> *held = nullptr) {
  constexpr int V = VecOf<S>::kN;
  const int lane = lane_id();
  uint32_t found = 0;
  uint32_t kept = 0;  // in `held`: the last ones found
  constexpr int64_t kStep = (int64_t)row<S>() * kRows;
  // Unaligned or held, the steps in flight are whole ones, and the rest of the stretch follows row by row: with the rows'
  // elements loaded one by one in this loop, 47 of its registers went to memory and were read again at every step
  // (62 M bf16 elements from an odd one on: 97 us, now 38; fp32, where they fitted, 84 and 61).
  const int64_t whole = ALIGNED && !HOLD ? end : begin + (end - begin) / kStep * kStep;
  auto load = [&](int64_t base, uint4 &a, uint4 &b, uint4 &c, uint4 &d) {
    if (!ALIGNED || HOLD || base + kStep <= end) {
      const S *at = in + base + lane * V;
      a = load16<S, ALIGNED, HOLD>(at);
      b = load16<S, ALIGNED, HOLD>(at + row<S>());
      c = load16<S, ALIGNED, HOLD>(at + 2 * row<S>());
      d = load16<S, ALIGNED, HOLD>(at + 3 * row<S>());
    } else {
      auto one = [&](int64_t first, uint4 &q) {
        S e[V];
        load_vec<S, ALIGNED>(in, first, end, e);  // past the end: zeros, never selected
        __builtin_memcpy(&q, e, 16);
      };
      one(base + lane * V, a);
      one(base + row<S>() + lane * V, b);
      one(base + 2 * row<S>() + lane * V, c);
      one(base + 3 * row<S>() + lane * V, d);
    }
  };
  auto write = [&](const uint4 &q, uint32_t bits, uint32_t pos, uint32_t first) {
    while (bits) {
      const uint32_t e = (uint32_t)__ffs((int)bits) - 1u;
      bits &= bits - 1u;
      if (pos < room) {
        *reinterpret_cast<I *>(reinterpret_cast<char *>(idx) + (uint32_t)(pos * sizeof(I))) = (I)(first + e);
        *reinterpret_cast<S *>(reinterpret_cast<char *>(val) + (uint32_t)(pos * sizeof(S))) = vec_pick(q, e, S(0));
      }
      ++pos;
    }
  };
  auto hold = [&](const uint4 &q, uint32_t bits, uint32_t pos, uint32_t first) {
    while (bits) {
      const uint32_t e = (uint32_t)__ffs((int)bits) - 1u;
      bits &= bits - 1u;
      held->idx[pos] = (int32_t)(first + e);
      held->val[pos] = vec_pick(q, e, S(0));
      ++pos;
    }
  };
  auto write_held = [&]() {
    __builtin_amdgcn_wave_barrier();
    for (uint32_t i = (uint32_t)lane; i < kept; i += 64u) {
      const uint32_t pos = found - kept + i;
      if (pos < room) {
        idx[pos] = (I)held->idx[i];
        val[pos] = held->val[i];
      }
    }
    __builtin_amdgcn_wave_barrier();
    kept = 0;
  };
  // two rows' counts in the halves of a word (a row has 512 elements at most)
  auto two = [&](const uint4 &q0, const uint4 &q1, uint32_t first) {
    const uint32_t x0 = vec_flags(q0, least, S(0)), x1 = vec_flags(q1, least, S(0));
    const uint32_t c = (uint32_t)__popc(x0) | ((uint32_t)__popc(x1) << 16);
    const uint32_t incl = wave_inclusive_scan(c);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    const uint32_t before = incl - c;
    if (HOLD) {
      static_assert(row<S>() <= (int)kHeld, "a row fits");
      if (kept + (total & 0xffffu) > kHeld) write_held();
      hold(q0, x0, kept + (before & 0xffffu), first);
      kept += total & 0xffffu;
      found += total & 0xffffu;
      if (kept + (total >> 16) > kHeld) write_held();
      hold(q1, x1, kept + (before >> 16), first + (uint32_t)row<S>());
      kept += total >> 16;
      found += total >> 16;
      return;
    }
    if (WRITE) {
      write(q0, x0, found + (before & 0xffffu), first);
      write(q1, x1, found + (total & 0xffffu) + (before >> 16), first + (uint32_t)row<S>());
    }
    found += (total & 0xffffu) + (total >> 16);
  };
  static_assert(kRows == 4, "four rows by name");
  uint4 a, b, c, d, na, nb, nc, nd;
  if (begin < whole) load(begin, na, nb, nc, nd);
#pragma unroll 1
  for (int64_t base = begin; base < whole; base += kStep) {
    a = na;
    b = nb;
    c = nc;
    d = nd;
    if (base + kStep < whole) load(base + kStep, na, nb, nc, nd);  // on its way while these rows are looked at
    const uint32_t first = (uint32_t)base + (uint32_t)(lane * V);
    two(a, b, first);
    two(c, d, first + 2u * (uint32_t)row<S>());
  }
  if constexpr (!ALIGNED || HOLD) {
#pragma unroll 1
    for (int64_t base = whole; base < end; base += row<S>()) {
      S e[V];
      load_vec<S, ALIGNED>(in, base + lane * V, end, e);
      uint4 q;
      __builtin_memcpy(&q, e, 16);
      two(q, make_uint4(0, 0, 0, 0), (uint32_t)base + (uint32_t)(lane * V));
    }
  }
  if (HOLD) write_held();
  return found;
}

__device__ inline uint32_t least_key(const uint32_t *thr, uint32_t mask) {
  uint32_t t = thr ? thr[0] : 1u;
  if (t == 0) t = 1;                 // zeros are never selected
  return t > mask ? mask + 1u : t;   // nothing qualifies
}

// Entries that still fit an output of `capacity` from place `at` on.
__device__ inline uint32_t room_from(int64_t capacity, uint64_t at) {
  const uint64_t left = at < (uint64_t)capacity ? (uint64_t)capacity - at : 0u;
  return left < 0xffffffffu ? (uint32_t)left : 0xffffffffu;
}

struct Stretches {
  int64_t len;      // elements of a stretch
  uint32_t count;   // stretches
  uint32_t quota;   // entries a stretch's part holds
  uint32_t *found;  // [count]
  int32_t *idx;     // [count * quota]
  void *val;
};

template <typename S>
Stretches plan_stretches(void *workspace, int64_t n, size_t *bytes) {
  Stretches st{};
  st.len = ceil_div(ceil_div(n > 0 ? n : 1, kMaxStretches), least_stretch<S>()) * least_stretch<S>();
  st.count = (uint32_t)ceil_div(n > 0 ? n : 1, st.len);
  st.quota = (uint32_t)(st.len / 8);
  Carver cv(workspace);
  if (n > kOneMax) {
    st.found = cv.take<uint32_t>(st.count);
    st.idx = cv.take<int32_t>((size_t)st.count * st.quota);
    st.val = cv.take<S>((size_t)st.count * st.quota);
  }
  *bytes = cv.used;
  return st;
}

template <typename S, bool ALIGNED>
__global__ __launch_bounds__(kBlock, 8) void k_compact_walk(const S *__restrict__ in, int64_t n,
                                                            const uint32_t *__restrict__ thr, Stretches st) {
  __shared__ Held<S> held[kBlock / 64];  // of a wave each
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t w = blockIdx.x * (uint32_t)(kBlock / 64) + wave;
  if (w >= st.count) return;
  const int64_t begin = (int64_t)w * st.len;
  const int64_t end = begin + st.len < n ? begin + st.len : n;
  const uint32_t found =
      walk<S, ALIGNED, true, true>(in, begin, end, least_key(thr, KeyOf<S>::kMask), st.idx + (size_t)w * st.quota,
                                   static_cast<S *>(st.val) + (size_t)w * st.quota, st.quota, &held[wave]);
  if (lane_id() == 0) st.found[w] = found;
}

// By the one thread that knows how many there are.  The host goes on from here, beside the move.
__device__ inline void count_known(uint64_t all, int64_t capacity, int64_t *out_count, const HostAnswer &answer,
                                   int32_t *status) {
  *out_count = (int64_t)all;
  int32_t bits = 0;
  if (all > (uint64_t)capacity) bits = atomicOr(status, ZEN_STAT_CAPACITY) | ZEN_STAT_CAPACITY;
  else if (answer.host) bits = __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!answer.host) return;
  host_store(answer.host + 1, (int64_t)all);
  host_store(answer.host + 2, (int64_t)bits);
  wait_global_acks();
  host_store(answer.host, answer.ticket);
}

template <typename S, typename I, bool ALIGNED>
__global__ __launch_bounds__(kMoveBlock) void k_compact_move(const S *__restrict__ in, int64_t n,
                                                             const uint32_t *__restrict__ thr, Stretches st,
                                                             I *__restrict__ out_idx, S *__restrict__ out_val,
                                                             int64_t capacity, int64_t *out_count, HostAnswer answer,
                                                             int32_t *status) {
  __shared__ uint32_t part[kMoveWaves];
  __shared__ uint32_t own[kMoveWaves];
  const uint32_t first = blockIdx.x * (uint32_t)kMoveWaves;
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t sum = 0;  // a tensor has fewer than 2^31 elements
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < first; i += kMoveBlock) sum += st.found[i];
  sum = wave_sum(sum);
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(first + wave));
  const uint32_t mine = w < st.count ? st.found[w] : 0u;
  if (lane_id() == 0) {
    part[wave] = sum;
    own[wave] = mine;
  }
  __syncthreads();
  uint64_t at = 0;
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kMoveWaves; ++i) at += part[i] + (i < wave ? own[i] : 0u);
  if (w + 1 == st.count && lane_id() == 0)
    count_known(at + mine, capacity, out_count, answer, status);
  if (w >= st.count) return;
  at = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32) |
       (uint32_t)__builtin_amdgcn_readfirstlane((int)at);  // the same in every lane
  if (mine > st.quota) {
    const int64_t begin = (int64_t)w * st.len;
    const int64_t end = begin + st.len < n ? begin + st.len : n;
    walk<S, ALIGNED, true>(in, begin, end, least_key(thr, KeyOf<S>::kMask), out_idx + at, out_val + at,
                           room_from(capacity, at));
    return;
  }
  const int32_t *idx = st.idx + (size_t)w * st.quota;
  const S *val = static_cast<const S *>(st.val) + (size_t)w * st.quota;
  constexpr int kAhead = 4;
  for (uint32_t i0 = 0; i0 < mine; i0 += 64 * kAhead) {
    int32_t k[kAhead];
    S v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const uint32_t i = i0 + (uint32_t)(j * 64 + lane_id());
      k[j] = idx[i < mine ? i : 0u];
      v[j] = val[i < mine ? i : 0u];
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const uint32_t i = i0 + (uint32_t)(j * 64 + lane_id());
      if (i < mine && at + i < (uint64_t)capacity) {
        out_idx[at + i] = (I)k[j];
        out_val[at + i] = v[j];
      }
    }
  }
}

template <typename S, typename I, bool ALIGNED>
__global__ __launch_bounds__(kMoveBlock) void k_compact_one(const S *__restrict__ in, int64_t n,
                                                            const uint32_t *__restrict__ thr, I *__restrict__ out_idx,
                                                            S *__restrict__ out_val, int64_t capacity,
                                                            int64_t *out_count, HostAnswer answer, int32_t *status) {
  __shared__ uint32_t own[kMoveWaves];
  const uint32_t wave = threadIdx.x >> 6;
  const uint32_t least = least_key(thr, KeyOf<S>::kMask);
  const int64_t len = (n + kMoveWaves * row<S>() - 1) / (kMoveWaves * row<S>()) * row<S>();
  const int64_t begin = (int64_t)wave * len < n ? (int64_t)wave * len : n;
  const int64_t end = begin + len < n ? begin + len : n;
  const uint32_t mine = walk<S, ALIGNED, false, false, I>(in, begin, end, least, nullptr, nullptr, 0);
  if (lane_id() == 0) own[wave] = mine;
  __syncthreads();
  uint64_t at = 0, all = 0;
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kMoveWaves; ++i) {
    at += i < wave ? own[i] : 0u;
    all += own[i];
  }
  if (threadIdx.x == 0) count_known(all, capacity, out_count, answer, status);
  at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);  // the same in every lane
  walk<S, ALIGNED, true>(in, begin, end, least, out_idx + at, out_val + at, room_from(capacity, at));
}

template <typename S, typename I, bool ALIGNED>
int compact_launch(const S *in, int64_t n, const uint32_t *thr, I *out_idx, S *out_val, int64_t capacity,
                   int64_t *out_count, void *workspace, int32_t *status, const HostAnswer &answer, hipStream_t s) {
  ProfScope prof(kProfSelectCompact, s);
  if (n <= kOneMax) {
    k_compact_one<S, I, ALIGNED><<<dim3(1), dim3(kMoveBlock), 0, s>>>(in, n, thr, out_idx, out_val, capacity, out_count,
                                                                     answer, status);
    ZEN_LAUNCH_CHECK("k_compact_one");
    return ZEN_OK;
  }
  size_t bytes;
  const Stretches st = plan_stretches<S>(workspace, n, &bytes);
  k_compact_walk<S, ALIGNED><<<dim3((unsigned)ceil_div(st.count, kBlock / 64)), dim3(kBlock), 0, s>>>(in, n, thr, st);
  ZEN_LAUNCH_CHECK("k_compact_walk");
  k_compact_move<S, I, ALIGNED><<<dim3((unsigned)ceil_div(st.count, kMoveWaves)), dim3(kMoveBlock), 0, s>>>(
      in, n, thr, st, out_idx, out_val, capacity, out_count, answer, status);
  ZEN_LAUNCH_CHECK("k_compact_move");
  return ZEN_OK;
}

template <typename S>
int compact_call(const void *input, int64_t n, const uint32_t *thr, void *out_idx, int idx64, void *out_val,
                 int64_t capacity, int64_t *out_count, void *workspace, int32_t *status, const HostAnswer &answer,
                 hipStream_t s) {
  const S *in = static_cast<const S *>(input);
  S *val = static_cast<S *>(out_val);
  const bool aligned = (reinterpret_cast<uintptr_t>(in) & 15u) == 0;
  if (idx64) {
    int64_t *idx = static_cast<int64_t *>(out_idx);
    return aligned ? compact_launch<S, int64_t, true>(in, n, thr, idx, val, capacity, out_count, workspace, status, answer, s)
                   : compact_launch<S, int64_t, false>(in, n, thr, idx, val, capacity, out_count, workspace, status, answer, s);
  }
  int32_t *idx = static_cast<int32_t *>(out_idx);
  return aligned ? compact_launch<S, int32_t, true>(in, n, thr, idx, val, capacity, out_count, workspace, status, answer, s)
                 : compact_launch<S, int32_t, false>(in, n, thr, idx, val, capacity, out_count, workspace, status, answer, s);
}

int select_call(const void *input, int dtype, int64_t n, const uint32_t *thr, void *out_idx, int idx64, void *out_val,
                int64_t capacity, int64_t *out_count, void *workspace, size_t workspace_bytes, int32_t *status,
                void *stream, const HostAnswer &answer = {}) {
  if (!out_count || !status) return fail(ZEN_EINVAL, "zen_select: null pointer");
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_select: bad dtype");
  if (n < 0 || n > 0x7fffffffll || capacity < 0) return fail(ZEN_EINVAL, "zen_select: need 0 <= n < 2^31");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n == 0) {
    launch_fill<int64_t>(out_count, 0, 1, s);
    ZEN_LAUNCH_CHECK("zen_select: zero count");
    return ZEN_OK;
  }
  if (!input || !workspace || (capacity > 0 && (!out_idx || !out_val)))
    return fail(ZEN_EINVAL, "zen_select: null pointer");
  if (workspace_bytes < zen_select_workspace(n, dtype)) return fail(ZEN_EWORKSPACE, "zen_select: workspace too small");
  if (dtype == ZEN_BF16)
    return compact_call<uint16_t>(input, n, thr, out_idx, idx64, out_val, capacity, out_count, workspace, status, answer, s);
  return compact_call<uint32_t>(input, n, thr, out_idx, idx64, out_val, capacity, out_count, workspace, status, answer, s);
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_select_workspace(int64_t n, int dtype) {
  size_t bytes;
  if (dtype == ZEN_BF16)
    (void)zen::plan_stretches<uint16_t>(nullptr, n, &bytes);
  else
    (void)zen::plan_stretches<uint32_t>(nullptr, n, &bytes);
  return bytes > 256 ? bytes : 256;
}

int zen_select(const void *input, int dtype, int64_t n, const uint32_t *thr, void *out_idx, int idx64,
               void *out_val, int64_t capacity, int64_t *out_count, void *workspace, size_t workspace_bytes,
               int32_t *status, void *stream) {
  return zen::select_call(input, dtype, n, thr, out_idx, idx64, out_val, capacity, out_count, workspace, workspace_bytes,
                          status, stream);
}

int zen_select_count(const void *input, int dtype, int64_t n, const uint32_t *thr, void *out_idx, int idx64,
                     void *out_val, int64_t capacity, int64_t *out_count, void *workspace, size_t workspace_bytes,
                     int32_t *status, int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  int rc = host_ask(host, words, 2, &answer);
  if (rc != ZEN_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = select_call(input, dtype, n, thr, out_idx, idx64, out_val, capacity, out_count, workspace, workspace_bytes,
                   status, stream, answer);
  if (rc == ZEN_OK && n == 0) rc = host_answer_launch(answer, out_count, 1, status, 1, s);
  return host_finish(rc, answer, s);
}

}  // extern "C"
