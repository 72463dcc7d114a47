// Second half of the sparse all-reduce with bitmaps, in one pass: every rank's bitmap over its partition's
// member list and its value list go straight into the dense gradient.  The reference turns each bitmap back
// into int64 indices by masking the cached member list (comm.py:87-99, 136-141) and scatter-adds all
// (index, value) lists into a zeroed dense tensor (comm.py:142-145, 32-44).  Neither the indices nor the
// member lists are needed for that: which partition an index belongs to is a hash away, and bit j of
// partition p's bitmap stands for the j-th index of that partition.  So the dense tensor is cut into tiles of
// 8192 indices; a dictionary built once per (numel, partitions) holds, per tile, the places of the tile's
// indices ordered by partition (16 bits each: partition 0's members in ascending order, then partition 1's,
// ...) and, per partition and tile, how many members lie below the tile.  A call first counts, per tile and
// partition, the set bits of the tile's bit range (which gives where the tile's values start in every value
// list); then a workgroup per tile brings the tile's bit ranges and values into LDS, looks up the place of
// every SET bit's member in the dictionary, and writes the tile once, zeros included: the dense tensor is
// never cleared, nothing is scattered in memory, and of the dictionary only the set bits' entries are read.
#include "zen_common.h"

namespace zen {
namespace {

constexpr int kFdTile = 8192;
constexpr int kFdBlock = 512;
constexpr int kFdPer = kFdTile / kFdBlock;   // consecutive indices per thread (16)
constexpr int kFdMaxLists = 64;
constexpr int kFdChunk = 16;                  // thread columns whose counts one thread adds up
constexpr int kFdChunks = kFdBlock / kFdChunk;
constexpr int kFdChunkRow = kFdChunks + 8;   // 16-bit words per list in the chunk table (rows stay 16-byte aligned)
static_assert(kFdChunks == 32, "a wave's lower half scans the chunk sums");

struct FdLists {
  const uint8_t *bitmap[kFdMaxLists];
  const void *val[kFdMaxLists];
  uint32_t bytes[kFdMaxLists], vals[kFdMaxLists];  // of the bitmap (2^28 at most: its bits fit 32 bits); values
};

__device__ inline uint32_t part_of(uint32_t t, uint32_t n, uint32_t npp) {
  return ((poly(t) + kSeed1) % n) / npp;  // functions_cuda_kernel.cu:172-175
}

// Dictionary, step 1: per tile the places of its indices ordered by partition, and the number of indices of
// every partition.  Dynamic LDS: P * (kFdBlock + kFdChunkRow) 16-bit counters.  Every thread counts, for its 16
// consecutive indices, how many belong to each list; prefix sums over the threads, in two levels (chunks of
// 16 threads, then the 32 chunks), give every index its rank inside its list.
__global__ __launch_bounds__(kFdBlock) void k_fd_order(uint32_t n, uint32_t npp, int P, uint16_t *__restrict__ order,
                                                      uint32_t *__restrict__ below) {
  extern __shared__ __attribute__((aligned(16))) uint16_t s_cnt[];  // [P][kFdBlock]
  uint16_t (*s_chunk)[kFdChunkRow] = reinterpret_cast<uint16_t (*)[kFdChunkRow]>(s_cnt + P * kFdBlock);  // [32]: the tile's total
  __shared__ uint32_t s_base[kFdMaxLists];  // members of lower lists in the tile
  const uint32_t tile_base = blockIdx.x * (uint32_t)kFdTile;
  const uint32_t base = tile_base + threadIdx.x * (uint32_t)kFdPer;
  uint32_t part[kFdPer];
#pragma unroll
  for (int e = 0; e < kFdPer; ++e) part[e] = base + e < n ? part_of(base + e, n, npp) : 0xffu;
  for (int p = 0; p < P; ++p) {
    uint32_t c = 0;
#pragma unroll
    for (int e = 0; e < kFdPer; ++e) c += part[e] == (uint32_t)p;
    s_cnt[p * kFdBlock + threadIdx.x] = (uint16_t)c;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < P * kFdChunks; q += kFdBlock) {
    const int p = q / kFdChunks, c = q % kFdChunks;
    uint16_t *col = s_cnt + p * kFdBlock + c * kFdChunk;
    uint32_t run = 0;
    for (int i = 0; i < kFdChunk; ++i) {
      const uint32_t x = col[i];
      col[i] = (uint16_t)run;
      run += x;
    }
    s_chunk[p][c] = (uint16_t)run;
  }
  __syncthreads();
  for (int p = threadIdx.x >> 6; p < P; p += kFdBlock / 64) {
    const int lane = lane_id();
    const uint32_t x = lane < kFdChunks ? s_chunk[p][lane] : 0u;
    const uint32_t incl = wave_inclusive_scan(x);
    if (lane < kFdChunks) s_chunk[p][lane] = (uint16_t)(incl - x);
    if (lane == kFdChunks - 1) s_chunk[p][kFdChunks] = (uint16_t)incl;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const uint32_t total = threadIdx.x < (uint32_t)P ? s_chunk[threadIdx.x][kFdChunks] : 0u;
    const uint32_t incl = wave_inclusive_scan(total);
    if (threadIdx.x < (uint32_t)P) {
      s_base[threadIdx.x] = incl - total;
      below[(size_t)blockIdx.x * P + threadIdx.x] = total;
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kFdPer; ++e) {
    const uint32_t p = part[e];
    if (p >= (uint32_t)P) continue;  // past the end of the tensor
    uint32_t rank = s_base[p] + s_chunk[p][threadIdx.x / kFdChunk] + s_cnt[p * kFdBlock + threadIdx.x];
#pragma unroll
    for (int f = 0; f < e; ++f) rank += part[f] == p;
    order[tile_base + rank] = (uint16_t)(threadIdx.x * kFdPer + e);
  }
}

// Per list (blockIdx.x): exclusive prefix over the tiles of a [tiles + 1][P] table of counts, in place; the last
// row receives the totals.  A thread takes eight consecutive tiles per round.  Run once per dictionary.
constexpr int kFdScanBlock = 1024;
constexpr int kFdScanPer = 8;
__global__ __launch_bounds__(kFdScanBlock) void k_fd_scan(uint32_t *__restrict__ table, uint32_t tiles, int P) {
  __shared__ uint32_t s_scan[kFdScanBlock / 64 + 1];
  uint32_t *column = table + blockIdx.x;
  uint32_t carry = 0;
  for (uint32_t base = 0; base < tiles; base += kFdScanBlock * kFdScanPer) {
    const uint32_t first = base + threadIdx.x * kFdScanPer;
    uint32_t c[kFdScanPer], sum = 0;
#pragma unroll
    for (int j = 0; j < kFdScanPer; ++j) {
      c[j] = first + j < tiles ? column[(size_t)(first + j) * P] : 0u;
      sum += c[j];
    }
    uint32_t total;
    uint32_t running = carry + block_exclusive_scan<uint32_t, kFdScanBlock>(sum, s_scan, &total);
#pragma unroll
    for (int j = 0; j < kFdScanPer; ++j) {
      if (first + j < tiles) column[(size_t)(first + j) * P] = running;
      running += c[j];
    }
    carry += total;
  }
  if (threadIdx.x == 0) column[(size_t)tiles * P] = carry;
}

// Set bits of bitmap `bm` in the bit range [b0, b1); bytes at or beyond `bytes` count as zero.  Read as
// aligned 64-bit words: a word that holds one byte of the bitmap lies in that byte's page, and what it holds
// beside the bitmap is masked away.
// AHEAD words are on their way at a time.
template <int AHEAD>
__device__ inline uint32_t popcount_range(const uint8_t *__restrict__ bm, int64_t bytes, uint32_t b0, uint32_t b1) {
  const uint64_t limit = (uint64_t)bytes * 8u;
  if (b1 > limit) b1 = (uint32_t)limit;
  if (b1 <= b0) return 0;
  const uintptr_t addr = reinterpret_cast<uintptr_t>(bm);
  const uint64_t *words = reinterpret_cast<const uint64_t *>(addr & ~(uintptr_t)7);
  const uint64_t lo = (uint64_t)b0 + (addr & 7u) * 8u, hi = (uint64_t)b1 + (addr & 7u) * 8u;  // bit numbers from words[0] on
  const uint64_t first = lo >> 6, last = (hi - 1u) >> 6;
  uint32_t c = 0;
  for (uint64_t w0 = first; w0 <= last; w0 += AHEAD) {
    unsigned long long x[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) x[j] = words[w0 + j <= last ? w0 + j : last];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const uint64_t w = w0 + j;
      if (w == first) x[j] &= ~0ull << (lo & 63u);
      if (w == last) x[j] &= ~0ull >> (63u - ((hi - 1u) & 63u));
      c += w <= last ? (uint32_t)__popcll(x[j]) : 0u;
    }
  }
  return c;
}

// Where the values of a tile start in every list, in two levels: the tiles are taken in groups of 256; a row of P
// words per tile holds the set bits of the group's tiles in front of it, a row per group the set bits in front of
// the group.
constexpr int kFdGroup = 256;
inline uint32_t fd_groups(uint32_t tiles) { return (tiles + kFdGroup - 1) / kFdGroup; }

// Per (group of tiles, list): set bits in each tile's bit range of the list's bitmap, summed up inside the
// group.  A bitmap shorter than its list (the reference's mask would not fit the member list, comm.py:97-98)
// raises ZEN_STAT_BAD_INDEX.
// A tile's range of a list spans eight or nine words at sixteen ranks (268 M elements: 22 us with one, 16 with five).
constexpr int kFdCountAhead = 5;
__global__ __launch_bounds__(kFdGroup) void k_fd_count(const uint32_t *__restrict__ below, uint32_t tiles, int P,
                                                       FdLists lists, uint32_t *__restrict__ vstart,
                                                       uint32_t *__restrict__ gsum, int32_t *status) {
  __shared__ uint32_t s_scan[kFdGroup / 64 + 1];
  const uint32_t tile = blockIdx.x * (uint32_t)kFdGroup + threadIdx.x;
  const int p = blockIdx.y;
  uint32_t cnt = 0;
  if (tile < tiles) {
    const size_t i = (size_t)tile * P + p;
    const uint32_t b0 = below[i], b1 = below[i + P];
    const int64_t bytes = lists.bytes[p];
    if (tile == tiles - 1 && ((int64_t)b1 + 7) / 8 > bytes) atomicOr(status, ZEN_STAT_BAD_INDEX);
    cnt = popcount_range<kFdCountAhead>(lists.bitmap[p], bytes, b0, b1);
  }
  uint32_t total;
  const uint32_t before = block_exclusive_scan<uint32_t, kFdGroup>(cnt, s_scan, &total);
  if (tile < tiles) vstart[(size_t)tile * P + p] = before;
  if (threadIdx.x == 0) gsum[(size_t)blockIdx.x * P + p] = total;
}

// Per list (blockIdx.x): exclusive prefix over the groups' sums, in place (a tensor of 2^31 elements has 1024 groups).
// A list with more set bits than values raises ZEN_STAT_BAD_INDEX.
constexpr int kFdGroupsMax = 1024;
__global__ __launch_bounds__(kFdGroupsMax) void k_fd_groups(uint32_t *__restrict__ gsum, uint32_t groups, int P, FdLists lists,
                                                            int32_t *status) {
  __shared__ uint32_t s_scan[kFdGroupsMax / 64 + 1];
  uint32_t *at = gsum + (size_t)threadIdx.x * P + blockIdx.x;
  const uint32_t v = threadIdx.x < groups ? *at : 0u;
  uint32_t total;
  const uint32_t before = block_exclusive_scan<uint32_t, kFdGroupsMax>(v, s_scan, &total);
  if (threadIdx.x < groups) *at = before;
  if (threadIdx.x == 0 && total > lists.vals[blockIdx.x]) atomicOr(status, ZEN_STAT_BAD_INDEX);
}

// Words of a chunk: sixteen lists have 512 members in a tile, few more than 576.  Tile kernel with 8, 9 and 10 words, us,
// 134 M bf16: 2 lists 171, 161 and 158, 3 185, 152 and 155, 4 176, 163 and 166, 8 184, 160 and 163, 16 190, 123 and 127,
// 24 156, 159 and 166, 32 190, 193 and 202, 64 318, 324 and 340; 67 M fp32: 2 112, 109 and 108, 4 124, 112 and 114, 16
// 132, 100 and 101, 64 195, 203 and 212.
constexpr int kFdWords = 9;
constexpr int kFdMembers = 64 * kFdWords;    // members of a chunk

template <typename S>
__device__ inline S fd_value(S v);  // what a zeroed element holds after one scatter_add_ of v (comm.py:35-39)
template <>
__device__ inline uint16_t fd_value<uint16_t>(uint16_t v) {  // 0.0f + v is v, but for -0 and signalling NaNs
  if (v == 0x8000u) v = 0;
  return (v & 0x7fffu) > 0x7f80u ? (uint16_t)(v | 0x40u) : v;
}
template <>
__device__ inline uint32_t fd_value<uint32_t>(uint32_t v) {
  return __float_as_uint(0.0f + __uint_as_float(v));
}

// fd_value of all elements of some pieces of a tile.  bf16 elements that need it are rare (-0 and NaNs), and three
// packed comparisons per pair find out that there is none.
template <int N>
__device__ inline void fd_values(u32x4 (&piece)[N], uint32_t) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) piece[i][e] = fd_value<uint32_t>(piece[i][e]);
}
template <int N>
__device__ inline void fd_values(u32x4 (&piece)[N], uint16_t) {
  typedef short i16x2 __attribute__((ext_vector_type(2)));
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  i16x2 most = {0, 0}, least = {0, 0};
  u16x2 top = {0, 0};
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t x = piece[i][e];
      most = __builtin_elementwise_max(most, __builtin_bit_cast(i16x2, x));
      least = __builtin_elementwise_min(least, __builtin_bit_cast(i16x2, x));
      top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, x));
    }
  // a NaN with a clear sign bit, -0, a NaN with the sign bit set
  if (most.x <= 0x7f80 && most.y <= 0x7f80 && least.x != -0x8000 && least.y != -0x8000 && top.x <= 0xff80 && top.y <= 0xff80)
    return;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      piece[i][e] = (uint32_t)fd_value<uint16_t>((uint16_t)piece[i][e]) |
                    (uint32_t)fd_value<uint16_t>((uint16_t)(piece[i][e] >> 16)) << 16;
}

// Lane i < kFdWords: bits [bit0 + 64 i, bit0 + 64 i + 64) of a bitmap of `limit` bits, from the two aligned words that
// hold them (a word with one byte of the bitmap lies in that byte's page); bits past `members` and past the bitmap's end
// are zero.
__device__ inline unsigned long long fd_chunk_bits(const uint8_t *bitmap, uint32_t limit, uint32_t bit0, uint32_t members) {
  const uintptr_t addr = reinterpret_cast<uintptr_t>(bitmap);
  const uint64_t *words = reinterpret_cast<const uint64_t *>(addr & ~(uintptr_t)7);
  const uint32_t first = bit0 + (uint32_t)(addr & 7u) * 8u;
  const uint32_t sh = first & 63u;
  const uint32_t has = bit0 < limit ? limit - bit0 : 0u;  // bits the bitmap has from the chunk's first on
  const uint32_t left = has < members ? has : members;
  const uint32_t lane = (uint32_t)lane_id();
  unsigned long long w = 0;
  if (lane * 64u < sh + left && left && lane <= (uint32_t)kFdWords) w = words[(first >> 6) + lane];
  const unsigned long long up = __shfl_down(w, 1, 64);
  unsigned long long bits = (w >> sh) | ((up << 1) << (63u - sh));
  if (lane >= (uint32_t)kFdWords || left <= lane * 64u) bits = 0;
  else if (left - lane * 64u < 64u) bits &= (1ull << (left - lane * 64u)) - 1ull;
  return bits;
}

// One workgroup per tile.  Lane p of every wave knows list p's members in the tile, the first bit of their range
// and where its values start; the lists' members are cut into chunks of 576, dealt to the waves in turn.  A
// wave gets the chunk's bits as nine 64-bit words in scalar registers: the word is the mask of the lanes whose
// member has a value, a lane's value is the one numbered by the set bits below it, and its place in the tile is
// the chunk's next entry of the dictionary, so that all loads are consecutive, nine of each kind in flight.  The
// places written are put together in LDS and leave with full-width stores.
// Bound by memory: two bytes of dictionary and one element of output per index, and the values.  62 M bf16 elements
// on sixteen ranks, 71 % of them set, 0.34 GB: 73 us; 268 M elements, 11 % set, 1.13 GB: 241 us, 4.7 TB/s.
// What a 64th of a chunk costs beside its loads counts too: places read without a look at the end of the list (the
// dictionary goes on behind it), values clamped only where they end, and 0.0f + v taken for what is written out as a
// whole instead of each value: 260 -> 249 us; chunks of nine words instead of ten, of which two were past most lists'
// ends, 241.  Slower: the bits by scalar loads (289; nine cache lines one after the other), the low bytes of the places
// alone with the high ones counted from where they wrap (0.86 GB, 275: seven instructions more per word).
// One SET bit per
// thread and turn, looked up in staged copies of the tile's bytes and values, took 307 and 411 us; with each value's
// load in a branch of its own, which makes the compiler wait for it there, this kernel took 129 and 428 (79 and 300 without).
// Waves of a workgroup meet at its two barriers, so small workgroups keep loads and stores going side by side as long
// as their tiles' LDS lets a compute unit hold enough of them: 16 KB a tile for bf16, four waves (the all-reduce of
// the 268 M elements 803 us; 837 with eight waves, 872 with two, 940 with sixteen), 32 KB for fp32, eight (200 M
// elements, two ranks: 865; 960 with four).
template <typename S>
constexpr int fd_tile_block() { return sizeof(S) == 2 ? 256 : 512; }

template <typename S>
__global__ __launch_bounds__(fd_tile_block<S>(), sizeof(S) == 2 ? 6 : 8) void k_fd_tiles(const uint16_t *__restrict__ order,
                                                       const uint32_t *__restrict__ below,
                                                       const uint32_t *__restrict__ vstart,
                                                       const uint32_t *__restrict__ gpre, int P, uint32_t n,
                                                       FdLists lists, S *__restrict__ dense, int32_t *status) {
  constexpr int kBlock = fd_tile_block<S>();
  __shared__ __attribute__((aligned(16))) S s_tile[kFdTile];
  const uint32_t tile = blockIdx.x;
  const uint32_t tile_base = tile * (uint32_t)kFdTile;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  uint32_t b0 = 0, b1 = 0, v0 = 0;
  if (lane < P) {
    const size_t at = (size_t)tile * P + lane;
    b0 = below[at];
    b1 = below[at + P];
    v0 = vstart[at] + gpre[(size_t)(tile / kFdGroup) * P + lane];
  }
  {
    uint4 *z = reinterpret_cast<uint4 *>(s_tile);
#pragma unroll
    for (int i = 0; i < (int)(kFdTile * sizeof(S) / 16) / kBlock; ++i) z[i * kBlock + threadIdx.x] = make_uint4(0, 0, 0, 0);
  }
  uint32_t cnt = b1 - b0;
  if (cnt > (uint32_t)kFdTile) cnt = 0;  // cannot be with a table this library built
  const uint32_t chunks = (cnt + kFdMembers - 1) / kFdMembers;
  const uint32_t incl = wave_inclusive_scan(cnt), cincl = wave_inclusive_scan(chunks);
  const uint32_t nchunks = (uint32_t)__builtin_amdgcn_readlane((int)cincl, 63);
  const bool odd = __builtin_amdgcn_readlane((int)incl, 63) > kFdTile;  // cannot be either
  __syncthreads();
#pragma unroll 1
  for (uint32_t c = (uint32_t)wave; c < nchunks && !odd; c += kBlock / 64) {
    const int p = (int)__popcll(__ballot(cincl <= c));  // the chunk's list
    const uint32_t j0 = (c - (uint32_t)__builtin_amdgcn_readlane((int)(cincl - chunks), p)) * kFdMembers;
    const uint32_t members = (uint32_t)__builtin_amdgcn_readlane((int)cnt, p) - j0;  // from here on, > 0
    const uint32_t bit0 = (uint32_t)__builtin_amdgcn_readlane((int)b0, p) + j0;
    const uint16_t *place_at = order + tile_base + (uint32_t)__builtin_amdgcn_readlane((int)(incl - cnt), p) + j0;
    uint32_t place[kFdWords];
#pragma unroll
    for (int i = 0; i < kFdWords; ++i)  // (past the members: the next list's, or what follows the last)
      place[i] = __builtin_nontemporal_load(place_at + lane + i * 64);
    const unsigned long long bits = fd_chunk_bits(lists.bitmap[p], lists.bytes[p] * 8u, bit0, members);
    // set bits of the tile's range in front of the chunk: the list's earlier chunks in this tile
    uint32_t nth = (uint32_t)__builtin_amdgcn_readlane((int)v0, p);
    if (j0) {  // 128 bits per lane
      const uint32_t from = bit0 - j0 + (uint32_t)lane * (kFdTile / 64);
      const uint32_t to = from + kFdTile / 64;
      nth += wave_sum(from < bit0 ? popcount_range<1>(lists.bitmap[p], lists.bytes[p], from, to < bit0 ? to : bit0) : 0u);
    }
    nth = (uint32_t)__builtin_amdgcn_readfirstlane((int)nth);
    const uint32_t have = lists.vals[p];
    unsigned long long word[kFdWords];
    uint32_t set = 0;
#pragma unroll
    for (int i = 0; i < kFdWords; ++i) {
      const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)bits, i);
      const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(bits >> 32), i);
      word[i] = ((unsigned long long)hi << 32) | lo;
      set += (uint32_t)__popcll(word[i]);
    }
    if (nth + set > have) {  // more set bits than values: the missing ones count as unset
      uint32_t front = 0;
      set = 0;
#pragma unroll
      for (int i = 0; i < kFdWords; ++i) {
        const uint32_t k = __builtin_amdgcn_mbcnt_hi((uint32_t)(word[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)word[i], front));
        front += (uint32_t)__popcll(word[i]);
        word[i] &= __ballot(nth + k < have);
        set += (uint32_t)__popcll(word[i]);
      }
    }
    if (set == 0) continue;
    // A member's value is the one numbered by the set bits below it.  The loads sit in no branch: lanes without a value
    // read that of the next that has one, or, at the end of all values, the last.
    const char *val = reinterpret_cast<const char *>(static_cast<const S *>(lists.val[p]) + nth);
    S v[kFdWords];
    uint32_t front = 0;
    if (nth + set < have) {
#pragma unroll
      for (int i = 0; i < kFdWords; ++i) {
        const uint32_t k = __builtin_amdgcn_mbcnt_hi((uint32_t)(word[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)word[i], front));
        v[i] = *reinterpret_cast<const S *>(val + (uint32_t)(k * sizeof(S)));
        front += (uint32_t)__popcll(word[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kFdWords; ++i) {
        const uint32_t k = __builtin_amdgcn_mbcnt_hi((uint32_t)(word[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)word[i], front));
        v[i] = *reinterpret_cast<const S *>(val + (uint32_t)((k < set ? k : set - 1u) * sizeof(S)));
        front += (uint32_t)__popcll(word[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kFdWords; ++i)
      if (__builtin_amdgcn_inverse_ballot_w64(word[i])) s_tile[place[i] & (uint32_t)(kFdTile - 1)] = v[i];
  }
  __syncthreads();
  // written out in 16-byte pieces, consecutive threads consecutive pieces: every store instruction fills whole lines
  if ((reinterpret_cast<uintptr_t>(dense) & 15u) == 0 && tile_base + (uint32_t)kFdTile <= n) {
    constexpr int kPieces = (int)(kFdTile * sizeof(S) / 16) / kBlock;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(s_tile);
    u32x4 *dst = reinterpret_cast<u32x4 *>(dense + tile_base);
    u32x4 piece[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) piece[i] = src[i * kBlock + threadIdx.x];
    fd_values(piece, S(0));
#pragma unroll
    for (int i = 0; i < kPieces; ++i) __builtin_nontemporal_store(piece[i], dst + i * kBlock + threadIdx.x);
  } else {
    for (uint32_t e = threadIdx.x; e < (uint32_t)kFdTile && tile_base + e < n; e += kBlock)
      dense[tile_base + e] = fd_value<S>(s_tile[e]);
  }
  if (odd && lane == 0) atomicOr(status, ZEN_STAT_BAD_INDEX);
}

inline uint32_t fd_tiles(int64_t numel) { return (uint32_t)ceil_div(numel, kFdTile); }
// (a chunk's places are read as if it were full)
inline size_t fd_order_bytes(int64_t numel) {
  return align_up(((size_t)fd_tiles(numel) * kFdTile + kFdMembers) * sizeof(uint16_t), 256);
}
inline size_t fd_table_bytes(int64_t numel, int P) { return align_up(((size_t)fd_tiles(numel) + 1) * P * sizeof(uint32_t), 256); }
inline size_t fd_vstart_bytes(int64_t numel, int P) { return align_up((size_t)fd_tiles(numel) * P * sizeof(uint32_t), 256); }
inline size_t fd_gsum_bytes(int64_t numel, int P) { return align_up((size_t)fd_groups(fd_tiles(numel)) * P * sizeof(uint32_t), 256); }

int fd_check(int64_t numel, int partitions) {
  if (numel <= 0 || numel > 0x7fffffffll || partitions < 1 || partitions > kFdMaxLists || numel / partitions == 0)
    return fail(ZEN_EINVAL, "zen_bitmap_dense: need 0 < partitions <= 64 and partitions <= numel < 2^31");
  return ZEN_OK;
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_bitmap_dense_dict_bytes(int64_t numel, int partitions) {
  if (zen::fd_check(numel, partitions) != ZEN_OK) return 0;
  return zen::fd_order_bytes(numel) + zen::fd_table_bytes(numel, partitions);
}

int zen_bitmap_dense_dict(int64_t numel, int partitions, void *dict, int64_t *members, void *stream) {
  using namespace zen;
  const int rc = fd_check(numel, partitions);
  if (rc != ZEN_OK) return rc;
  if (!dict || (reinterpret_cast<uintptr_t>(dict) & 15u)) return fail(ZEN_EINVAL, "zen_bitmap_dense_dict: null or unaligned dictionary");
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint16_t *order = static_cast<uint16_t *>(dict);
  uint32_t *below = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(dict) + fd_order_bytes(numel));
  const uint32_t tiles = fd_tiles(numel);
  const size_t lds = (size_t)partitions * (kFdBlock + kFdChunkRow) * sizeof(uint16_t);
  if (lds > 32768)  // beyond what a launch may ask for without saying so first
    ZEN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_fd_order), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_fd_order<<<dim3(tiles), dim3(kFdBlock), lds, s>>>((uint32_t)numel, (uint32_t)(numel / partitions), partitions, order, below);
  ZEN_LAUNCH_CHECK("k_fd_order");
  k_fd_scan<<<dim3((unsigned)partitions), dim3(kFdScanBlock), 0, s>>>(below, tiles, partitions);
  ZEN_LAUNCH_CHECK("k_fd_scan");
  if (members) {  // the list lengths, for a caller that sizes bitmaps without a mapping
    for (int p = 0; p < partitions; ++p) members[p] = 0;
    ZEN_HIP_CHECK(hipStreamSynchronize(s));
    uint32_t host[kFdMaxLists];
    for (int p = 0; p < partitions; ++p) {
      ZEN_HIP_CHECK(hipMemcpy(&host[p], below + (size_t)tiles * partitions + p, sizeof(uint32_t), hipMemcpyDeviceToHost));
      members[p] = host[p];
    }
  }
  return ZEN_OK;
}

size_t zen_bitmap_dense_workspace(int64_t numel, int partitions) {
  if (zen::fd_check(numel, partitions) != ZEN_OK) return 0;
  return zen::fd_vstart_bytes(numel, partitions) + zen::fd_gsum_bytes(numel, partitions);
}

int zen_bitmap_dense_lists(const void *dict, int64_t numel, int partitions, const uint8_t *const *bitmaps,
                           const int64_t *bitmap_bytes, const void *const *values, int dtype,
                           const int64_t *value_count, void *dense, void *workspace, size_t workspace_bytes,
                           int32_t *status, void *stream) {
  using namespace zen;
  const int rc = fd_check(numel, partitions);
  if (rc != ZEN_OK) return rc;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_bitmap_dense: bad dtype");
  if (!dict || !bitmaps || !bitmap_bytes || !values || !value_count || !dense || !workspace || !status)
    return fail(ZEN_EINVAL, "zen_bitmap_dense: null pointer");
  if (workspace_bytes < zen_bitmap_dense_workspace(numel, partitions))
    return fail(ZEN_EWORKSPACE, "zen_bitmap_dense: workspace too small");
  FdLists lists{};
  for (int p = 0; p < partitions; ++p) {
    if (bitmap_bytes[p] < 0 || value_count[p] < 0) return fail(ZEN_EINVAL, "zen_bitmap_dense: negative length");
    if ((bitmap_bytes[p] > 0 && !bitmaps[p]) || (value_count[p] > 0 && !values[p]))
      return fail(ZEN_EINVAL, "zen_bitmap_dense: null pointer");
    // what lies beyond the members a list can have is never looked at
    lists.bitmap[p] = bitmaps[p];
    lists.bytes[p] = (uint32_t)(bitmap_bytes[p] < (1ll << 28) ? bitmap_bytes[p] : 1ll << 28);
    lists.val[p] = values[p];
    lists.vals[p] = (uint32_t)(value_count[p] < (1ll << 31) ? value_count[p] : 1ll << 31);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t *order = static_cast<const uint16_t *>(dict);
  const uint32_t *below = reinterpret_cast<const uint32_t *>(static_cast<const uint8_t *>(dict) + fd_order_bytes(numel));
  uint32_t *vstart = static_cast<uint32_t *>(workspace);
  uint32_t *gsum = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(workspace) + fd_vstart_bytes(numel, partitions));
  const uint32_t tiles = fd_tiles(numel);
  const uint32_t groups = fd_groups(tiles);
  ProfScope prof(kProfDecodeFused, s);
  k_fd_count<<<dim3(groups, (unsigned)partitions), dim3(kFdGroup), 0, s>>>(below, tiles, partitions, lists, vstart, gsum,
                                                                       status);
  ZEN_LAUNCH_CHECK("k_fd_count");
  k_fd_groups<<<dim3((unsigned)partitions), dim3(kFdGroupsMax), 0, s>>>(gsum, groups, partitions, lists, status);
  ZEN_LAUNCH_CHECK("k_fd_groups");
  if (dtype == ZEN_BF16)
    k_fd_tiles<uint16_t><<<dim3(tiles), dim3(fd_tile_block<uint16_t>()), 0, s>>>(order, below, vstart, gsum, partitions, (uint32_t)numel,
                                                                lists, static_cast<uint16_t *>(dense), status);
  else
    k_fd_tiles<uint32_t><<<dim3(tiles), dim3(fd_tile_block<uint32_t>()), 0, s>>>(order, below, vstart, gsum, partitions, (uint32_t)numel,
                                                                lists, static_cast<uint32_t *>(dense), status);
  ZEN_LAUNCH_CHECK("k_fd_tiles");
  return ZEN_OK;
}

int zen_bitmap_dense_lists_status(const void *dict, int64_t numel, int partitions, const uint8_t *const *bitmaps,
                                  const int64_t *bitmap_bytes, const void *const *values, int dtype,
                                  const int64_t *value_count, void *dense, void *workspace, size_t workspace_bytes,
                                  int32_t *status, int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  HostAnswer answer;
  int rc = host_ask(host, words, 1, &answer);
  if (rc != ZEN_OK) return rc;
  rc = zen_bitmap_dense_lists(dict, numel, partitions, bitmaps, bitmap_bytes, values, dtype, value_count, dense, workspace,
                              workspace_bytes, status, stream);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (rc == ZEN_OK) rc = host_answer_launch(answer, nullptr, 0, status, 1, s);
  return host_finish(rc, answer, s);
}

int zen_bitmap_dense(const void *dict, int64_t numel, int partitions, const uint8_t *bitmaps,
                     const int64_t *bitmap_start, const void *values, int dtype, const int64_t *value_start,
                     void *dense, void *workspace, size_t workspace_bytes, int32_t *status, void *stream) {
  using namespace zen;
  const int rc = fd_check(numel, partitions);
  if (rc != ZEN_OK) return rc;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_bitmap_dense: bad dtype");
  if (!bitmap_start || !value_start) return fail(ZEN_EINVAL, "zen_bitmap_dense: null pointer");
  const uint8_t *bitmap_at[kFdMaxLists];
  const void *value_at[kFdMaxLists];
  int64_t bytes[kFdMaxLists], vals[kFdMaxLists];
  for (int p = 0; p < partitions; ++p) {
    bytes[p] = bitmap_start[p + 1] - bitmap_start[p];
    vals[p] = value_start[p + 1] - value_start[p];
    if (bytes[p] < 0 || vals[p] < 0) return fail(ZEN_EINVAL, "zen_bitmap_dense: list offsets must not decrease");
    if ((bytes[p] > 0 && !bitmaps) || (vals[p] > 0 && !values)) return fail(ZEN_EINVAL, "zen_bitmap_dense: null pointer");
    bitmap_at[p] = bitmaps + bitmap_start[p];
    value_at[p] = static_cast<const char *>(values) + value_start[p] * (dtype == ZEN_BF16 ? 2 : 4);
  }
  return zen_bitmap_dense_lists(dict, numel, partitions, bitmap_at, bytes, value_at, dtype, vals, dense, workspace,
                                workspace_bytes, status, stream);
}

}  // extern "C"
