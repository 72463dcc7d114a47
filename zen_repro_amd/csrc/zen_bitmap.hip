// Bitmap index codec of the second exchange (comm.py:59-99): a rank describes
// which members of its partition's ascending index list are present by one bit
// per member, least significant bit first inside each byte.
//
// Encode is a lookup per index.  A rank dictionary kept next to the mapping
// (members below every multiple of 96, plus one membership bit per index
// value) answers it with one load; without the dictionary the position is
// estimated by interpolation (the members are spread evenly, that is what the
// hash is for), bracketed by doubling steps and found by bisection.  Decode is a compaction of the set bits: count per
// block, scan the block counts, write mapping[position] for every set bit.
#include "zen_common.h"

namespace zen {
namespace {

constexpr int kBmBlock = 256;
constexpr int kBmBytes = 16;                       // bitmap bytes per thread in decode
constexpr int kBmSpan = kBmBlock * kBmBytes * 8;   // positions per workgroup (32768)

// First position whose member is >= v (torch.searchsorted, left; comm.py:61), looked for around position g:
// doubling steps away from g until v is bracketed, then bisection inside the bracket.
__device__ inline int64_t member_lower_bound_near(const int64_t *__restrict__ map, int64_t count, int64_t g,
                                                  int64_t step, int64_t v) {
  int64_t lo, hi;  // map[lo] < v (lo = -1: nothing below), map[hi] >= v (hi = count: nothing at or above)
  if (map[g] < v) {
    lo = g;
    hi = g + step;
    while (hi < count && map[hi] < v) {
      lo = hi;
      step <<= 1;
      hi += step;
    }
    if (hi > count) hi = count;
  } else {
    hi = g;
    lo = g - step;
    while (lo >= 0 && map[lo] >= v) {
      hi = lo;
      step <<= 1;
      lo -= step;
    }
    if (lo < -1) lo = -1;
  }
  while (hi - lo > 1) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (map[mid] < v)
      lo = mid;
    else
      hi = mid;
  }
  return hi;
}

// Rank dictionary of one partition's member list, kept next to the list: per 96 index values, 16 bytes with the number
// of members below them and their membership bits.  The position of any index is then that number plus the set bits
// below its own: one load that neighbouring indices share, a sixth of a byte per index value, instead of a search
// through eight-byte members.  (Blocks of 512 bits with their ranks in an array of their own are an eighth of a byte, but
// sixteen words to mask and count per index: the marking kernel 21.5 us where it takes 12.)
constexpr uint32_t kBmValues = 96;

// One thread per block: a bisection for its first member, which the others follow in the list.
__global__ __launch_bounds__(kBmBlock) void k_bitmap_ranks(const int64_t *__restrict__ map, int64_t count,
                                                           int64_t blocks, uint4 *__restrict__ ranks) {
  const int64_t b = (int64_t)blockIdx.x * kBmBlock + threadIdx.x;
  if (b >= blocks) return;
  const int64_t v = b * kBmValues;
  int64_t lo = -1, hi = count;
  while (hi - lo > 1) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (map[mid] < v)
      lo = mid;
    else
      hi = mid;
  }
  uint32_t w[kBmValues / 32] = {};
  for (int64_t j = hi; j < count && map[j] < v + kBmValues; ++j) {
    const uint32_t off = (uint32_t)(map[j] - v);
#pragma unroll
    for (uint32_t q = 0; q < kBmValues / 32; ++q) w[q] |= (off >> 5) == q ? 1u << (off & 31) : 0u;
  }
  ranks[b] = make_uint4((uint32_t)hi, w[0], w[1], w[2]);
}

// Index v's place among the members (`count`: behind the last).
// Without the dictionary the position is estimated by interpolation over the whole list (the members are
// spread evenly, that is what the hash is for; float arithmetic lands within a few thousand places) and
// corrected by a search around the estimate.
__device__ inline int64_t member_place(const int64_t *__restrict__ map, int64_t count, int64_t v) {
  const int64_t first = map[0], last = map[count - 1];
  if (v <= first) return 0;
  if (v > last) return count;
  const float slope = (float)(count - 1) / (float)(last - first);
  int64_t g = (int64_t)((float)(v - first) * slope);
  g = g > count - 1 ? count - 1 : (g < 0 ? 0 : g);
  return member_lower_bound_near(map, count, g, 64, v);
}

// kBmEach indices per thread, those of a wave's row neighbours; the indices may come in any order.  Bound by the trips
// to memory (the index, the dictionary's line, the bitmap's word), of which
// four of each kind are in flight.  2.8 M of the 3.9 M members of a sixteenth of 62 M indices 12.0 us, 2.1 M of the
// 16.8 M of 268 M 13.9; with one index per thread, lines of 512 membership bits and the neighbours' bits gathered
// through lane permutes 25.9 and 22.8.  (One, two, eight indices per thread: 14.0, 13.2, 14.0 and 13.7, 13.8, 15.0.)
constexpr int kBmEach = 4;
template <typename I, bool RANKS>
__global__ __launch_bounds__(kBmBlock, 4) void k_bitmap_mark(const int64_t *__restrict__ map, int64_t count,
                                                             const I *__restrict__ idx, int64_t idx_n,
                                                             const int64_t *__restrict__ idx_n_dev,
                                                             const uint4 *__restrict__ ranks, int64_t numel,
                                                             uint32_t *__restrict__ words, int32_t *status) {
  int64_t n = idx_n;
  if (idx_n_dev) {
    const int64_t d = *idx_n_dev;
    n = d < n ? (d < 0 ? 0 : d) : n;
  }
  if (count <= 0) {
    if (n > 0 && blockIdx.x == 0 && threadIdx.x == 0) atomicOr(status, ZEN_STAT_BAD_INDEX);
    return;
  }
  const int64_t j0 = (int64_t)blockIdx.x * (kBmBlock * kBmEach) + threadIdx.x;
  if (j0 - (int64_t)threadIdx.x >= n) return;
  int64_t v[kBmEach];
  uint32_t pos[kBmEach];  // below 2^31
#pragma unroll
  for (int i = 0; i < kBmEach; ++i) {  // (a place past the end reads the last index and marks nothing)
    const int64_t j = j0 + i * kBmBlock;
    v[i] = (int64_t)idx[j < n ? j : n - 1];
  }
  if (RANKS) {
    uint4 entry[kBmEach];
#pragma unroll
    for (int i = 0; i < kBmEach; ++i)  // in no branch, so that all are in flight together
      entry[i] = ranks[v[i] < 0 || v[i] >= numel ? 0u : (uint32_t)v[i] / kBmValues];
#pragma unroll
    for (int i = 0; i < kBmEach; ++i) {
      const uint32_t off = (uint32_t)v[i] % kBmValues;
      const uint32_t below = (1u << (off & 31u)) - 1u;  // of the bits in the index's own word
      const uint32_t all = entry[i].x + (uint32_t)__popc(entry[i].y & (off < 32u ? below : ~0u)) +
                           (uint32_t)__popc(off < 32u ? 0u : entry[i].z & (off < 64u ? below : ~0u)) +
                           (uint32_t)__popc(off < 64u ? 0u : entry[i].w & below);
      // an index beyond the index range is beyond every member
      pos[i] = v[i] < 0 ? 0u : v[i] >= numel ? (uint32_t)count : all;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kBmEach; ++i) pos[i] = (uint32_t)member_place(map, count, v[i]);
  }
  // Neighbouring lanes often mark the same word (ascending indices: positions a few places apart): of the lanes that
  // do, the last one goes to memory.
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < kBmEach; ++i) {
    const bool live = j0 + i * kBmBlock < n;
    const bool bad = !live || pos[i] >= (uint32_t)count;
    if (live && bad) atomicOr(status, ZEN_STAT_BAD_INDEX);  // torch raises an index error here (comm.py:63)
    const uint32_t word = bad ? 0xffffffffu : pos[i] >> 5;
    uint32_t bits = bad ? 0u : 1u << (pos[i] & 31u);
    const uint32_t prev = (uint32_t)__shfl_up((int)word, 1), before = (uint32_t)__shfl_up((int)pos[i], 1);
    const uint64_t starts = __ballot(lane == 0 || word != prev);  // stretches of lanes that name one word
    if (__ballot(lane > 0 && !bad && before >= pos[i])) {
      // not strictly ascending: a lane gathers the bits of the lanes before it that name the same word.  (It may also
      // pick up bits of the same word from further away: harmless for an OR.)
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t w2 = (uint32_t)__shfl_up((int)word, off);
        const uint32_t b2 = (uint32_t)__shfl_up((int)bits, off);
        if (lane >= off && w2 == word) bits |= b2;
      }
    } else {
      // all bits of a stretch are different: their OR is their sum
      const uint32_t upto = wave_inclusive_scan(bits);
      const int first = 63 - __clzll((long long)(starts & (~0ull >> (63 - lane))));
      bits = upto - (uint32_t)__shfl((int)(upto - bits), first);
    }
    if (!bad && (lane == 63 || ((starts >> lane) & 2ull))) atomicOr(&words[word], bits);
  }
}

template <typename I>
void launch_mark(const int64_t *map, int64_t count, const I *idx, int64_t idx_n, const int64_t *idx_n_dev,
                 const uint32_t *rank_at, int64_t numel, uint32_t *words, int32_t *status, hipStream_t s) {
  const auto kernel = rank_at ? k_bitmap_mark<I, true> : k_bitmap_mark<I, false>;
  kernel<<<dim3((unsigned)ceil_div(idx_n, (int64_t)kBmBlock * kBmEach)), dim3(kBmBlock), 0, s>>>(
      map, count, idx, idx_n, idx_n_dev, reinterpret_cast<const uint4 *>(rank_at), numel, words, status);
}

// Bits of the 16 bitmap bytes of thread t of block b that lie below `count` positions, as four words.
__device__ inline void load_bits(const uint8_t *__restrict__ bitmap, int64_t bytes, int64_t count, int64_t byte0,
                                 uint32_t (&w)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t x = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t at = byte0 + q * 4 + e;
      if (at < bytes) x |= (uint32_t)bitmap[at] << (8 * e);
    }
    const int64_t pos0 = (byte0 + q * 4) * 8;  // position of bit 0 of this word
    if (pos0 >= count)
      x = 0;
    else if (count - pos0 < 32)
      x &= (1u << (count - pos0)) - 1u;
    w[q] = x;
  }
}

__global__ __launch_bounds__(kBmBlock) void k_bitmap_count(const uint8_t *__restrict__ bitmap, int64_t bytes,
                                                           int64_t count, uint32_t *__restrict__ partial) {
  __shared__ uint32_t s_scan[kBmBlock / 64];
  uint32_t w[4];
  load_bits(bitmap, bytes, count, ((int64_t)blockIdx.x * kBmBlock + threadIdx.x) * kBmBytes, w);
  const uint32_t c = (uint32_t)(__popc(w[0]) + __popc(w[1]) + __popc(w[2]) + __popc(w[3]));
  uint32_t total;
  block_exclusive_scan<uint32_t, kBmBlock>(c, s_scan, &total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// One workgroup: partial[b] becomes the number of set bits before block b; the total goes to *out_count.
__global__ __launch_bounds__(1024) void k_bitmap_scan(uint32_t *__restrict__ partial, uint32_t blocks,
                                                      int64_t capacity, int64_t *__restrict__ out_count,
                                                      int32_t *status) {
  __shared__ uint64_t s_scan[1024 / 64];
  __shared__ uint64_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  for (uint32_t base = 0; base < blocks; base += 1024) {
    const uint32_t b = base + threadIdx.x;
    const uint64_t c = b < blocks ? partial[b] : 0;
    uint64_t total;
    const uint64_t before = block_exclusive_scan<uint64_t, 1024>(c, s_scan, &total);
    const uint64_t carry = s_carry;
    // the offsets stay below 2^32: a bitmap describes fewer than 2^31 positions
    if (b < blocks) partial[b] = (uint32_t)(carry + before);
    __syncthreads();
    if (threadIdx.x == 0) s_carry = carry + total;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *out_count = (int64_t)s_carry;
    if ((int64_t)s_carry > capacity) atomicOr(status, ZEN_STAT_CAPACITY);
  }
}

constexpr int kBmList = 4096;  // set bits a workgroup hands on per round

// The positions of the set bits go through a list in LDS, in order: consecutive threads then fetch
// consecutive entries (loads that do not wait for each other) and write consecutive outputs.
__global__ __launch_bounds__(kBmBlock) void k_bitmap_emit(const int64_t *__restrict__ map,
                                                          const uint8_t *__restrict__ bitmap, int64_t bytes,
                                                          int64_t count, const uint32_t *__restrict__ partial,
                                                          int64_t *__restrict__ out, int64_t capacity) {
  __shared__ uint32_t s_scan[kBmBlock / 64];
  __shared__ uint32_t s_pos[kBmList];
  uint32_t w[4];
  const int64_t byte0 = ((int64_t)blockIdx.x * kBmBlock + threadIdx.x) * kBmBytes;
  load_bits(bitmap, bytes, count, byte0, w);
  const uint32_t c = (uint32_t)(__popc(w[0]) + __popc(w[1]) + __popc(w[2]) + __popc(w[3]));
  uint32_t total;
  const uint32_t mine = block_exclusive_scan<uint32_t, kBmBlock>(c, s_scan, &total);
  const int64_t base = (int64_t)partial[blockIdx.x];
  const int64_t pos0 = (int64_t)blockIdx.x * kBmSpan;  // first position of this workgroup
  for (uint32_t round = 0; round < total; round += kBmList) {
    uint32_t at = mine;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t x = w[q];
      while (x) {
        const int bit = __ffs((int)x) - 1;
        x &= x - 1;
        if (at - round < (uint32_t)kBmList) s_pos[at - round] = threadIdx.x * (kBmBytes * 8) + q * 32 + bit;
        ++at;
      }
    }
    __syncthreads();
    const uint32_t here = total - round < (uint32_t)kBmList ? total - round : (uint32_t)kBmList;
    for (uint32_t e = threadIdx.x; e < here; e += kBmBlock) {
      const int64_t o = base + round + e;
      if (o < capacity) out[o] = map[pos0 + s_pos[e]];
    }
    __syncthreads();
  }
}

inline int64_t decode_blocks(int64_t count) { return ceil_div(count > 0 ? count : 1, kBmSpan); }

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_bitmap_words(int64_t mapping_n) { return mapping_n > 0 ? (size_t)((mapping_n + 31) / 32) : 0; }

size_t zen_bitmap_rank_words(int64_t numel) {
  if (numel <= 0) return 0;
  return (size_t)zen::ceil_div(numel, (int64_t)zen::kBmValues) * 4;
}

int zen_bitmap_ranks(const int64_t *mapping_p, int64_t mapping_n, int64_t numel, uint32_t *rank_at, void *stream) {
  using namespace zen;
  if (mapping_n < 0 || mapping_n > 0x7fffffffll || numel <= 0 || numel > 0x7fffffffll)
    return fail(ZEN_EINVAL, "zen_bitmap_ranks: need 0 < numel < 2^31");
  if (!rank_at || (mapping_n > 0 && !mapping_p)) return fail(ZEN_EINVAL, "zen_bitmap_ranks: null pointer");
  if (reinterpret_cast<uintptr_t>(rank_at) & 15u) return fail(ZEN_EINVAL, "zen_bitmap_ranks: table not 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t blocks = ceil_div(numel, (int64_t)kBmValues);
  k_bitmap_ranks<<<dim3((unsigned)ceil_div(blocks, kBmBlock)), dim3(kBmBlock), 0, s>>>(mapping_p, mapping_n, blocks,
                                                                                     reinterpret_cast<uint4 *>(rank_at));
  ZEN_LAUNCH_CHECK("k_bitmap_ranks");
  return ZEN_OK;
}

int zen_bitmap_encode(const int64_t *mapping_p, int64_t mapping_n, const void *idx, int idx64, int64_t idx_n,
                      const int64_t *idx_n_dev, const uint32_t *rank_at, int64_t numel, uint32_t *bitmap_words,
                      int32_t *status, void *stream) {
  using namespace zen;
  if (mapping_n < 0 || mapping_n > 0x7fffffffll || idx_n < 0) return fail(ZEN_EINVAL, "zen_bitmap_encode: bad size");
  if (!status || (mapping_n > 0 && (!mapping_p || !bitmap_words)) || (idx_n > 0 && !idx))
    return fail(ZEN_EINVAL, "zen_bitmap_encode: null pointer");
  if (rank_at && (numel <= 0 || numel > 0x7fffffffll || (reinterpret_cast<uintptr_t>(rank_at) & 15u)))
    return fail(ZEN_EINVAL, "zen_bitmap_encode: a rank dictionary needs its numel (below 2^31) and 16-byte alignment");
  if (reinterpret_cast<uintptr_t>(bitmap_words) & 3u) return fail(ZEN_EINVAL, "zen_bitmap_encode: bitmap not 4-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  launch_fill<uint32_t>(bitmap_words, 0u, zen_bitmap_words(mapping_n), s);
  ZEN_LAUNCH_CHECK("zen_bitmap_encode: clear");
  if (idx_n == 0) return ZEN_OK;
  if (ceil_div(idx_n, kBmBlock) > 0x7fffffffll) return fail(ZEN_EINVAL, "zen_bitmap_encode: too many indices");
  if (idx64)
    launch_mark(mapping_p, mapping_n, static_cast<const int64_t *>(idx), idx_n, idx_n_dev, rank_at, numel, bitmap_words,
                status, s);
  else
    launch_mark(mapping_p, mapping_n, static_cast<const int32_t *>(idx), idx_n, idx_n_dev, rank_at, numel, bitmap_words,
                status, s);
  ZEN_LAUNCH_CHECK("k_bitmap_mark");
  return ZEN_OK;
}

int zen_bitmap_encode_status(const int64_t *mapping_p, int64_t mapping_n, const void *idx, int idx64, int64_t idx_n,
                             const int64_t *idx_n_dev, const uint32_t *rank_at, int64_t numel, uint32_t *bitmap_words,
                             int32_t *status, int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  int rc = host_ask(host, words, 1, &answer);
  if (rc != ZEN_OK) return rc;
  rc = zen_bitmap_encode(mapping_p, mapping_n, idx, idx64, idx_n, idx_n_dev, rank_at, numel, bitmap_words, status, stream);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (rc == ZEN_OK) rc = host_answer_launch(answer, nullptr, 0, status, 1, s);
  return host_finish(rc, answer, s);
}

size_t zen_bitmap_decode_workspace(int64_t mapping_n) {
  return zen::align_up((size_t)zen::decode_blocks(mapping_n) * sizeof(uint32_t), 256);
}

int zen_bitmap_decode(const int64_t *mapping_p, int64_t mapping_n, const uint8_t *bitmap, int64_t bitmap_bytes,
                      int64_t *out, int64_t capacity, int64_t *out_count, void *workspace, size_t workspace_bytes,
                      int32_t *status, void *stream) {
  using namespace zen;
  if (mapping_n < 0 || mapping_n > 0x7fffffffll || capacity < 0 || bitmap_bytes < 0)
    return fail(ZEN_EINVAL, "zen_bitmap_decode: bad size");
  if (bitmap_bytes < (mapping_n + 7) / 8)  // the reference's mask would be shorter than the list it indexes
    return fail(ZEN_EINVAL, "zen_bitmap_decode: bitmap shorter than the mapping");
  if (!out_count || !status || !workspace || (mapping_n > 0 && (!mapping_p || !bitmap)) || (capacity > 0 && !out))
    return fail(ZEN_EINVAL, "zen_bitmap_decode: null pointer");
  if (workspace_bytes < zen_bitmap_decode_workspace(mapping_n))
    return fail(ZEN_EWORKSPACE, "zen_bitmap_decode: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint32_t *partial = static_cast<uint32_t *>(workspace);
  const int64_t blocks = decode_blocks(mapping_n);
  k_bitmap_count<<<dim3((unsigned)blocks), dim3(kBmBlock), 0, s>>>(bitmap, bitmap_bytes, mapping_n, partial);
  ZEN_LAUNCH_CHECK("k_bitmap_count");
  k_bitmap_scan<<<dim3(1), dim3(1024), 0, s>>>(partial, (uint32_t)blocks, capacity, out_count, status);
  ZEN_LAUNCH_CHECK("k_bitmap_scan");
  k_bitmap_emit<<<dim3((unsigned)blocks), dim3(kBmBlock), 0, s>>>(mapping_p, bitmap, bitmap_bytes, mapping_n, partial,
                                                                 out, capacity);
  ZEN_LAUNCH_CHECK("k_bitmap_emit");
  return ZEN_OK;
}

}  // extern "C"
