// Dense decode of payloads that arrive as ascending lists (zen_decode_dense_sorted).
//
// The second exchange of the sparse all-reduce hands every rank all ranks'
// merged shards, each an ascending index list, and the reference scatter-adds
// them into a zeroed dense tensor (comm.py:142-145 with :32-44); method 1 does
// the same with every rank's own ascending selection (comm.py:113-117).  A
// dense result needs no sort: the dense tensor is cut into tiles of kDecTile
// elements, a first kernel finds where every tile starts in every list, and one
// workgroup per tile gathers its entries (a contiguous stretch of every list)
// into a copy of the tile in LDS and writes the tile out with full-width
// stores.  The dense tensor is written exactly once and never cleared first.
//
// Sums are taken in fp32 from +0 in payload order and rounded once, like
// zen_decode_dense: inside a list every index occurs once (the lists are
// strictly ascending; that is checked), so a tile whose entries are all
// distinct takes them in any order, and a tile in which two lists meet on an
// index goes through the lists one after the other.
#include "zen_common.h"

namespace zen {
namespace {

constexpr int kDecTile = 8192;   // dense elements per workgroup (its LDS copy: 16 KB for bf16, 32 KB for fp32)
constexpr int kDecBlock = 512;   // four workgroups fill a compute unit's wave slots; 34 KB of LDS each
constexpr int kDecMaxLists = 64;
constexpr int kDecLanes = 4;     // entries per lane in flight
constexpr int kDecChunk = 64 * kDecLanes;  // entries of one list a wave takes at a time

struct DecLists {
  const void *idx[kDecMaxLists];
  const void *val[kDecMaxLists];
  uint32_t len[kDecMaxLists];
  int n;
};

// Number of entries of the list with index < t * kDecTile (by a search that assumes the list ascending; the tile kernel
// checks that it is).  Bound by the memory lines it asks for, one for nearly
// every probe: a list that a hash chose is spread evenly, so the place is guessed from the key and then from what
// was found at the guess, a little further than needed so that the answer gets bracketed from both sides; a
// handful of probes leaves a stretch inside a line or two, which is bisected (any list is, after kDecGuesses
// probes).  Sixteen lists of 1.8 M entries, 7564 tiles: 13 us, bisection alone 27.
constexpr int kDecGuesses = 6;
constexpr uint32_t kDecNear = 16;
template <typename I>
__device__ inline uint32_t decode_start(const I *__restrict__ list, uint32_t len, int64_t t, int64_t ntiles, int64_t dense_n) {
  uint32_t lo = 0, hi = len;  // the answer lies in [lo, hi]
  if (t == 0 || len == 0) {
    hi = 0;
  } else if (t == ntiles) {
    lo = len;
  } else {
    const int64_t key = t * (int64_t)kDecTile;
    const float per = (float)len / (float)dense_n;  // entries per index
    float guess = (float)key * per;
    for (int i = 0; i < kDecGuesses && hi - lo > kDecNear; ++i) {
      uint32_t g = guess > (float)lo ? (uint32_t)guess : lo;
      if (g >= hi) g = hi - 1u;
      const int64_t k = (int64_t)list[g];
      if (k < key) lo = g + 1u; else hi = g;
      const float d = (float)(key - k) * per;  // entries between here and there
      const float more = 3.0f + 0.5f * sqrtf(fabsf(d));
      guess = (float)g + d + (k < key ? more : -more);
    }
    while (lo < hi) {
      const uint32_t mid = lo + ((hi - lo) >> 1);
      if ((int64_t)list[mid] < key) lo = mid + 1u; else hi = mid;
    }
  }
  return lo;
}

// Up to so many tiles, one to a compute unit, search for themselves: a launch less, for a chain of probes in every tile
// (bf16, a call with the search in the tiles / in a kernel in front: two lists into 9000 elements 22.2 / 25.2 us, four
// into a million 24.2 / 26.2, sixteen of a tenth of two million 44.7 / 47.8).
constexpr int64_t kDecFew = 256;

// starts[l * (ntiles + 1) + t]: decode_start of list l.
template <typename I>
__global__ __launch_bounds__(256) void k_decode_starts(DecLists lists, int64_t ntiles, int64_t dense_n,
                                                       uint32_t *__restrict__ starts) {
  const int l = blockIdx.y;
  const int64_t t = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (t > ntiles) return;
  starts[(int64_t)l * (ntiles + 1) + t] =
      decode_start(static_cast<const I *>(lists.idx[l]), lists.len[l], t, ntiles, dense_n);
}

// The value a dense element gets from one entry: +0 + v in fp32, rounded to the tensor's type (-0 becomes +0,
// like in a scatter_add_ into zeros).
__device__ inline uint16_t single_value(uint16_t v) { return f32_to_bf16_rne(0.0f + KeyOf<uint16_t>::to_f32(v)); }
__device__ inline uint32_t single_value(uint32_t v) { return __float_as_uint(0.0f + __uint_as_float(v)); }
__device__ inline uint16_t rounded(float f, uint16_t) { return f32_to_bf16_rne(f); }
__device__ inline uint32_t rounded(float f, uint32_t) { return __float_as_uint(f); }

// 16 bytes of output: the tensor's elements [first, first + V), as wide as its end and alignment allow.
template <typename S>
__device__ inline void store_vec(const S (&e)[16 / sizeof(S)], S *__restrict__ dense, int64_t first, int64_t dense_n,
                                 bool aligned) {
  constexpr int V = 16 / sizeof(S);
  if (aligned && first + V <= dense_n) {
    u32x4 q;
    __builtin_memcpy(&q, e, 16);
    __builtin_nontemporal_store(q, reinterpret_cast<u32x4 *>(dense + first));
  } else {
#pragma unroll
    for (int q = 0; q < V; ++q)
      if (first + q < dense_n) dense[first + q] = e[q];
  }
}

// One workgroup per tile.  Anything that contradicts "every list strictly ascending, every index inside
// [0, dense_n)" raises ZEN_STAT_RETRY (the caller repeats with zen_decode_dense, which takes any input).
// Bound by the trips to memory of a tile, of which there are three: the lists' stretches, the entries, the
// output.  Lane l of every wave knows list l's stretch; the stretches are cut into chunks of 256 entries of one
// list, dealt to the eight waves in turn, so that a wave's loads are consecutive, four of them per lane are in
// flight and no entry has to look for its list.  (Entries numbered through and dealt to threads one by one, each
// bisecting for its list and waiting for its own load: 182 us for 28.7 M entries of sixteen lists into 62 M bf16
// elements, now 80.)
// FEW: the tile finds its stretches itself, two waves for both ends.
template <typename I, typename S, bool FEW>
__global__ __launch_bounds__(kDecBlock) void k_decode_tiles(DecLists lists, int64_t ntiles,
                                                            const uint32_t *__restrict__ starts,
                                                            S *__restrict__ dense, int64_t dense_n, int32_t *status) {
  // the tile in the tensor's own type or, where lists meet, as fp32 sums
  __shared__ __attribute__((aligned(16))) float acc[kDecTile];
  __shared__ uint32_t occ[kDecTile / 32];
  __shared__ uint32_t s_count, s_wrong;
  static_assert(kDecMaxLists == 64 && kDecTile / 32 <= kDecBlock, "a list per lane, a word of occ per thread");
  S *tile = reinterpret_cast<S *>(acc);
  constexpr int V = 16 / (int)sizeof(S);
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t = blockIdx.x;
  const int64_t first = t * (int64_t)kDecTile;
  __shared__ uint32_t s_ends[FEW ? 2 : 1][64];
  uint32_t a = 0, b = 0;  // asked for first: the answer is on its way while the tile is cleared
  if (FEW) {
    if (wave < 2 && lane < lists.n)
      s_ends[wave][lane] = decode_start(static_cast<const I *>(lists.idx[lane]), lists.len[lane], t + wave, ntiles, dense_n);
  } else if (lane < lists.n) {
    const uint32_t *at = starts + (int64_t)lane * (ntiles + 1) + t;
    a = at[0];
    b = at[1];
  }
  for (int j = tid; j < kDecTile * (int)sizeof(S) / 16; j += kDecBlock)
    reinterpret_cast<uint4 *>(acc)[j] = make_uint4(0, 0, 0, 0);
  if (tid < kDecTile / 32) occ[tid] = 0;
  if (tid == 0) s_count = s_wrong = 0;
  if (FEW) {
    __syncthreads();
    if (lane < lists.n) {
      a = s_ends[0][lane];
      b = s_ends[FEW ? 1 : 0][lane];
    }
  }
  bool wrong = b < a;  // the search went astray: the list is not ascending
  const uint32_t len = wrong ? 0u : b - a;
  const uint32_t chunks = (len + kDecChunk - 1) / kDecChunk;
  const uint32_t cincl = wave_inclusive_scan(chunks), lincl = wave_inclusive_scan(len);
  const uint32_t nchunks = (uint32_t)__builtin_amdgcn_readlane((int)cincl, 63);
  const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)lincl, 63);
  __syncthreads();
  for (uint32_t c = (uint32_t)wave; c < nchunks; c += kDecBlock / 64) {
    const int l = (int)__popcll(__ballot(cincl <= c));  // the chunk's list
    const uint32_t la = (uint32_t)__builtin_amdgcn_readlane((int)a, l);
    const uint32_t lb = (uint32_t)__builtin_amdgcn_readlane((int)b, l);
    const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)(cincl - chunks), l);
    const uint32_t e0 = la + (c - before) * kDecChunk;  // < lb
    const I *idx = static_cast<const I *>(lists.idx[l]);
    const S *val = static_cast<const S *>(lists.val[l]);
    I k[kDecLanes];
    S v[kDecLanes];
#pragma unroll
    for (int i = 0; i < kDecLanes; ++i) {
      const uint32_t e = e0 + (uint32_t)(i * 64 + lane);
      k[i] = idx[e < lb ? e : lb - 1u];
      v[i] = val[e < lb ? e : lb - 1u];
    }
    int64_t prev = e0 > 0 ? (int64_t)idx[e0 - 1u] : -1;  // the entry before it in its list must be smaller
#pragma unroll
    for (int i = 0; i < kDecLanes; ++i) {
      const uint32_t e = e0 + (uint32_t)(i * 64 + lane);
      const int64_t up = (int64_t)__shfl_up(k[i], 1, 64);
      const int64_t left = lane == 0 ? prev : up;
      prev = (int64_t)__shfl(k[i], 63, 64);
      const uint64_t off = (uint64_t)((int64_t)k[i] - first);
      const bool bad = off >= (uint64_t)kDecTile || (int64_t)k[i] >= dense_n || left >= (int64_t)k[i];
      if (e < lb) {
        if (bad) {
          wrong = true;
        } else {
          atomicOr(&occ[off >> 5], 1u << (off & 31u));
          tile[off] = single_value(v[i]);
        }
      }
    }
  }
  if (wrong) s_wrong = 1;
  __syncthreads();
  if (s_wrong) {
    if (tid == 0) atomicOr(status, ZEN_STAT_RETRY);
    return;  // the caller repeats the whole call: what this tile holds does not matter
  }
  {  // as many different elements as entries?
    const uint32_t mine = wave_sum(tid < kDecTile / 32 ? (uint32_t)__popc(occ[tid]) : 0u);
    if (lane == 0 && mine) atomicAdd(&s_count, mine);
  }
  __syncthreads();
  const bool aligned = (reinterpret_cast<uintptr_t>(dense + first) & 15u) == 0;
  if (s_count == total) {
    for (int j = tid * V; j < kDecTile; j += kDecBlock * V) {
      S e[V];
      const uint4 q = *reinterpret_cast<const uint4 *>(tile + j);
      __builtin_memcpy(e, &q, 16);
      store_vec<S>(e, dense, first + j, dense_n, aligned);
    }
    return;
  }
  // Two lists share an index here: fp32 sums, the lists one after the other (inside a list every index occurs
  // once).  The entries are fetched again (they are in the caches), those of kAhead lists at a time.
  __syncthreads();
  for (int j = tid; j < kDecTile / 4; j += kDecBlock) reinterpret_cast<uint4 *>(acc)[j] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  constexpr int kAhead = 8;
  // What lists with nothing in the tile read: the tiles' starts, or where there are none an entry of some list (which has to
  // be found first: 250 M bf16 elements, four lists of 1 %, 241 us instead of 231; 89 M, eight of 5 %, 154 and 145).
  const I *no_idx = reinterpret_cast<const I *>(starts);
  const S *no_val = reinterpret_cast<const S *>(starts);
  if (FEW) {
    const int other = __ffsll((unsigned long long)__ballot(a < b)) - 1;
    const uint32_t other_at = (uint32_t)__builtin_amdgcn_readlane((int)a, other);
    no_idx = static_cast<const I *>(lists.idx[other]) + other_at;
    no_val = static_cast<const S *>(lists.val[other]) + other_at;
  }
  for (int l0 = 0; l0 < lists.n; l0 += kAhead) {
    // an entry of each list per thread, in no branch (a list with nothing for this thread reads some entry), so
    // that all are in flight together
    I k[kAhead];
    S v[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int l = l0 + i < lists.n ? l0 + i : lists.n - 1;
      const uint32_t la = (uint32_t)__builtin_amdgcn_readlane((int)a, l);
      const uint32_t lb = (uint32_t)__builtin_amdgcn_readlane((int)b, l);
      const bool some = la < lb;
      const I *idx = some ? static_cast<const I *>(lists.idx[l]) + la : no_idx;
      const S *val = some ? static_cast<const S *>(lists.val[l]) + la : no_val;
      const uint32_t e = la + (uint32_t)tid < lb ? (uint32_t)tid : 0u;
      k[i] = idx[e];
      v[i] = val[e];
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (l0 + i < lists.n) {
        const uint32_t la = (uint32_t)__builtin_amdgcn_readlane((int)a, l0 + i);
        const uint32_t lb = (uint32_t)__builtin_amdgcn_readlane((int)b, l0 + i);
        if (la + (uint32_t)tid < lb) acc[(uint32_t)((int64_t)k[i] - first)] += KeyOf<S>::to_f32(v[i]);
        for (uint32_t e = la + (uint32_t)(tid + kDecBlock); e < lb; e += kDecBlock)
          acc[(uint32_t)((int64_t) static_cast<const I *>(lists.idx[l0 + i])[e] - first)] +=
              KeyOf<S>::to_f32(static_cast<const S *>(lists.val[l0 + i])[e]);
        __syncthreads();
      }
    }
  }
  for (int j = tid * V; j < kDecTile; j += kDecBlock * V) {
    S e[V];
#pragma unroll
    for (int q = 0; q < V; ++q) e[q] = rounded(acc[j + q], S(0));
    store_vec<S>(e, dense, first + j, dense_n, aligned);
  }
}

template <typename I, typename S>
int decode_sorted_launch(const DecLists &lists, void *dense, int64_t dense_n, uint32_t *starts, int32_t *status,
                         hipStream_t s) {
  const int64_t ntiles = ceil_div(dense_n, (int64_t)kDecTile);
  S *out = static_cast<S *>(dense);
  if (ntiles <= kDecFew) {
    k_decode_tiles<I, S, true><<<dim3((unsigned)ntiles), dim3(kDecBlock), 0, s>>>(lists, ntiles, nullptr, out, dense_n, status);
  } else {
    k_decode_starts<I><<<dim3((unsigned)ceil_div(ntiles + 1, (int64_t)256), (unsigned)lists.n), dim3(256), 0, s>>>(
        lists, ntiles, dense_n, starts);
    ZEN_LAUNCH_CHECK("k_decode_starts");
    k_decode_tiles<I, S, false><<<dim3((unsigned)ntiles), dim3(kDecBlock), 0, s>>>(lists, ntiles, starts, out, dense_n, status);
  }
  ZEN_LAUNCH_CHECK("k_decode_tiles");
  return ZEN_OK;
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_decode_dense_sorted_workspace(int64_t dense_n, int nlists) {
  if (dense_n <= 0 || nlists <= 0) return 256;
  const int64_t ntiles = zen::ceil_div(dense_n, (int64_t)zen::kDecTile);
  return (size_t)((ntiles + 1) * nlists) * sizeof(uint32_t) + 256;
}

int zen_decode_dense_lists(const void *const *idx, int idx64_in, const void *const *val, int dtype, const int64_t *len,
                           int nlists, void *dense, int64_t dense_n, void *workspace, size_t workspace_bytes,
                           int32_t *status, void *stream) {
  using namespace zen;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_decode_dense_lists: bad dtype");
  if (!dense || !status || !idx || !val || !len || !workspace)
    return fail(ZEN_EINVAL, "zen_decode_dense_lists: null pointer");
  if (nlists < 1 || nlists > kDecMaxLists) return fail(ZEN_EINVAL, "zen_decode_dense_lists: 1 to 64 lists");
  if (dense_n <= 0 || dense_n > 0x7fffffff00ll) return fail(ZEN_EINVAL, "zen_decode_dense_lists: bad dense size");
  DecLists lists{};
  lists.n = nlists;
  for (int l = 0; l < nlists; ++l) {
    if (len[l] < 0 || len[l] > 0xfffff000ll)
      return fail(ZEN_EINVAL, "zen_decode_dense_lists: lists hold fewer than 2^32 entries");
    if (len[l] > 0 && (!idx[l] || !val[l])) return fail(ZEN_EINVAL, "zen_decode_dense_lists: null pointer");
    lists.idx[l] = idx[l];
    lists.val[l] = val[l];
    lists.len[l] = (uint32_t)len[l];
  }
  if (workspace_bytes < zen_decode_dense_sorted_workspace(dense_n, nlists))
    return fail(ZEN_EWORKSPACE, "zen_decode_dense_lists: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint32_t *starts = static_cast<uint32_t *>(workspace);
  if (dtype == ZEN_BF16)
    return idx64_in ? decode_sorted_launch<int64_t, uint16_t>(lists, dense, dense_n, starts, status, s)
                    : decode_sorted_launch<int32_t, uint16_t>(lists, dense, dense_n, starts, status, s);
  return idx64_in ? decode_sorted_launch<int64_t, uint32_t>(lists, dense, dense_n, starts, status, s)
                  : decode_sorted_launch<int32_t, uint32_t>(lists, dense, dense_n, starts, status, s);
}

int zen_decode_dense_lists_status(const void *const *idx, int idx64_in, const void *const *val, int dtype, const int64_t *len,
                                  int nlists, void *dense, int64_t dense_n, void *workspace, size_t workspace_bytes,
                                  int32_t *status, int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  int rc = host_ask(host, words, 1, &answer);
  if (rc != ZEN_OK) return rc;
  rc = zen_decode_dense_lists(idx, idx64_in, val, dtype, len, nlists, dense, dense_n, workspace, workspace_bytes, status, stream);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (rc == ZEN_OK) rc = host_answer_launch(answer, nullptr, 0, status, 1, s);
  return host_finish(rc, answer, s);
}

int zen_decode_dense_sorted(const void *idx, int idx64_in, const void *val, int dtype, const int64_t *list_start,
                            int nlists, void *dense, int64_t dense_n, void *workspace, size_t workspace_bytes,
                            int32_t *status, void *stream) {
  using namespace zen;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_decode_dense_sorted: bad dtype");
  if (!dense || !status || !list_start || !workspace) return fail(ZEN_EINVAL, "zen_decode_dense_sorted: null pointer");
  if (nlists < 1 || nlists > kDecMaxLists) return fail(ZEN_EINVAL, "zen_decode_dense_sorted: 1 to 64 lists");
  const void *idx_at[kDecMaxLists], *val_at[kDecMaxLists];
  int64_t len[kDecMaxLists];
  for (int l = 0; l < nlists; ++l) {
    if (list_start[l] < 0 || list_start[l + 1] < list_start[l])
      return fail(ZEN_EINVAL, "zen_decode_dense_sorted: list offsets must ascend (lists below 2^32 entries)");
    idx_at[l] = static_cast<const char *>(idx) + list_start[l] * (idx64_in ? 8 : 4);
    val_at[l] = static_cast<const char *>(val) + list_start[l] * (dtype == ZEN_BF16 ? 2 : 4);
    len[l] = list_start[l + 1] - list_start[l];
  }
  if (list_start[0] != 0) return fail(ZEN_EINVAL, "zen_decode_dense_sorted: the first list starts at 0");
  if (list_start[nlists] > 0 && (!idx || !val)) return fail(ZEN_EINVAL, "zen_decode_dense_sorted: null pointer");
  return zen_decode_dense_lists(idx_at, idx64_in, val_at, dtype, len, nlists, dense, dense_n, workspace,
                                workspace_bytes, status, stream);
}

}  // extern "C"
