// Second half of the sparse all-reduce with bitmaps, in one pass: every rank's bitmap over its partition's
// member list and its value list go straight into the dense gradient.  The reference turns each bitmap back
// into int64 indices by masking the cached member list (comm.py:87-99, 136-141) and scatter-adds all
// (index, value) lists into a zeroed dense tensor (comm.py:142-145, 32-44).  Neither the indices nor the
// member lists are needed for that: which partition an index belongs to is a hash away, and bit j of
// partition p's bitmap stands for the j-th index of that partition.  So the dense tensor is cut into tiles; a
// dictionary built once per (numel, partitions) holds, per tile, the places of the tile's indices ordered by
// partition (partition 0's members in ascending order, then partition 1's, ...; up to sixteen partitions a byte
// each, the distance from the member in front, else 16 bits) and, per partition and tile, how many members lie
// below the tile.  A call first counts, per tile and partition, the set bits of the tile's bit range (which gives
// where the tile's values start in every value list); then a workgroup per tile puts the values in their members'
// places in LDS and writes the tile once, zeros included: the dense tensor is never cleared and nothing is
// scattered in memory.
#include <type_traits>

#include "zen_common.h"

namespace zen {
namespace {

constexpr int kFdTile = 8192;
constexpr int kFdBlock = 512;
constexpr int kFdMaxLists = 64;

// Dictionaries of bytes: a member's place is that of the member in front of it in its list plus a byte, which takes half
// the memory of places of 16 bits.  The members of a list lie as far apart as there are lists, give or take: up to
// sixteen lists one distance in ten million does not fit a byte (its chunk's word holds it), at 32 lists one in three
// thousand and at 64 one in fifty, so that nearly every tile would have some.  A lane takes eight members, a chunk is
// what a wave takes, and seven eighths of 8192 elements to a tile keep the lists' shares under whole chunks: at sixteen
// lists 448 members, give or take 20.
constexpr int kFdByteLists = 16;
constexpr int kFdByteTile = 7168;
constexpr int kFdLane = 8;                               // members a lane takes
constexpr int kFdByteChunk = 64 * kFdLane;
constexpr int kFdByteRow = kFdByteTile + kFdLane * kFdByteLists;  // bytes of a tile: lists begin at multiples of kFdLane
constexpr int kFdByteChunks = 32;                        // words of a tile's chunk table
// A chunk's word: the place of its first member; kFdFar if another of its members lies 256 or more behind the one in front
// of it (its byte is zero), and in the upper half how far; kFdSeveral if more than one does.
constexpr uint32_t kFdPlace = 0x1fffu, kFdFar = 0x8000u, kFdSeveral = 0x4000u;
static_assert(kFdByteTile / kFdByteChunk + kFdByteLists <= kFdByteChunks, "every chunk of a tile has a word");
static_assert(kFdByteTile % (16 * kFdBlock / 64) == 0 && kFdByteTile <= (int)kFdPlace + 1 && kFdByteRow % 16 == 0, "tile layout");
constexpr int kFdChunk = 16;                  // thread columns whose counts one thread adds up
constexpr int kFdChunks = kFdBlock / kFdChunk;
constexpr int kFdChunkRow = kFdChunks + 8;   // 16-bit words per list in the chunk table (rows stay 16-byte aligned)
static_assert(kFdChunks == 32, "a wave's lower half scans the chunk sums");

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct FdLists {
  const uint8_t *bitmap[kFdMaxLists];
  const void *val[kFdMaxLists];
  uint32_t bytes[kFdMaxLists], vals[kFdMaxLists];  // of the bitmap (2^28 at most: its bits fit 32 bits); values
};

// Division by a number known to the host: its inverse, rounded down, gives the quotient or one less.
struct FdDivisor {
  uint32_t d, inverse;  // floor(2^32 / d), or 2^32 - 1
};
inline FdDivisor fd_divisor(uint32_t d) { return {d, d > 1 ? (uint32_t)((1ull << 32) / d) : 0xffffffffu}; }
__device__ inline uint32_t part_of(uint32_t t, FdDivisor n, FdDivisor npp) {  // hash % n / npp, functions_cuda_kernel.cu:172-175
  const uint32_t h = poly(t) + kSeed1;
  uint32_t rem = h - __umulhi(h, n.inverse) * n.d;  // below 2 n
  if (rem >= n.d) rem -= n.d;
  const uint32_t part = __umulhi(rem, npp.inverse);
  return part + (rem - part * npp.d >= npp.d ? 1u : 0u);
}

// Dictionary, step 1: per tile the places of its indices ordered by partition, and the number of indices of
// every partition.  Every thread counts, for its consecutive indices, how many belong to each list; prefix sums over
// the threads, in two levels (chunks of 16 threads, then the 32 chunks), give every index its rank inside its list.
// BYTES: `order` holds distances (kFdByteRow bytes a tile, lists padded to whole lanes; a chunk's first is one) and
// chunk_at a word per chunk of a list's members (kFdPlace).  Else 16-bit places, kFdTile a tile.  Dynamic LDS: fd_order_lds.
template <bool BYTES>
__global__ __launch_bounds__(kFdBlock) void k_fd_order(FdDivisor n, FdDivisor npp, int P, void *__restrict__ order,
                                                      uint32_t *__restrict__ chunk_at, uint32_t *__restrict__ below) {
  constexpr int kTile = BYTES ? kFdByteTile : kFdTile;
  constexpr int kPer = kTile / kFdBlock;  // consecutive indices per thread
  extern __shared__ __attribute__((aligned(16))) uint16_t s_cnt[];  // [P][kFdBlock]
  uint16_t (*s_chunk)[kFdChunkRow] = reinterpret_cast<uint16_t (*)[kFdChunkRow]>(s_cnt + P * kFdBlock);  // [32]: the tile's total
  __shared__ uint32_t s_base[kFdMaxLists];   // where a list begins in the tile's row
  __shared__ uint32_t s_first[kFdMaxLists];  // BYTES: chunks of lower lists
  const uint32_t tile_base = blockIdx.x * (uint32_t)kTile;
  const uint32_t base = tile_base + threadIdx.x * (uint32_t)kPer;
  uint32_t part[kPer];
#pragma unroll
  for (int e = 0; e < kPer; ++e) part[e] = base + e < n.d ? part_of(base + e, n, npp) : 0xffu;
  uint32_t rank[kPer];  // among the thread's own, for now
  if constexpr (BYTES) {
    // four bits a list (268 M elements on sixteen lists: 810 us with a comparison per element and list and per pair of
    // elements, and with the compiler's divisions; 570 so)
    static_assert(kPer < 16 && kFdByteLists <= 16, "counters of four bits");
    uint64_t count = 0;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      const uint32_t at = part[e] * 4u & 63u;
      rank[e] = (uint32_t)(count >> at) & 15u;
      count += (uint64_t)(part[e] < (uint32_t)P ? 1u : 0u) << at;
    }
    for (int p = 0; p < P; ++p) s_cnt[p * kFdBlock + threadIdx.x] = (uint16_t)((uint32_t)(count >> (4 * p)) & 15u);
  } else {
    for (int p = 0; p < P; ++p) {
      uint32_t c = 0;
#pragma unroll
      for (int e = 0; e < kPer; ++e) c += part[e] == (uint32_t)p;
      s_cnt[p * kFdBlock + threadIdx.x] = (uint16_t)c;
    }
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      rank[e] = 0;
#pragma unroll
      for (int f = 0; f < e; ++f) rank[e] += part[f] == part[e];
    }
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
    const uint32_t room = BYTES ? (total + kFdLane - 1) / kFdLane * kFdLane : total;
    const uint32_t chunks = (total + kFdByteChunk - 1) / kFdByteChunk;
    const uint32_t incl = wave_inclusive_scan(room), cincl = wave_inclusive_scan(chunks);
    if (threadIdx.x < (uint32_t)P) {
      s_base[threadIdx.x] = incl - room;
      s_first[threadIdx.x] = cincl - chunks;
      below[(size_t)blockIdx.x * P + threadIdx.x] = total;
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const uint32_t p = part[e];
    if (p >= (uint32_t)P) continue;  // past the end of the tensor
    rank[e] += s_chunk[p][threadIdx.x / kFdChunk] + s_cnt[p * kFdBlock + threadIdx.x];
    if (!BYTES) static_cast<uint16_t *>(order)[tile_base + s_base[p] + rank[e]] = (uint16_t)(threadIdx.x * kPer + e);
  }
  if constexpr (BYTES) {
    uint16_t *s_place = &s_chunk[P][0];                                   // [kFdByteRow]
    uint8_t *s_byte = reinterpret_cast<uint8_t *>(s_place + kFdByteRow);  // [kFdByteRow]
    __shared__ uint32_t s_at[kFdByteChunks], s_far[kFdByteChunks];
    if (threadIdx.x < kFdByteChunks) s_at[threadIdx.x] = s_far[threadIdx.x] = 0;
    // what pads a list to whole lanes belongs to nobody
    for (int i = threadIdx.x; i < kFdByteRow / 4; i += kFdBlock) reinterpret_cast<uint32_t *>(s_byte)[i] = 0x01010101u;
#pragma unroll
    for (int e = 0; e < kPer; ++e)
      if (part[e] < (uint32_t)P) s_place[s_base[part[e]] + rank[e]] = (uint16_t)(threadIdx.x * kPer + e);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      const uint32_t p = part[e];
      if (p >= (uint32_t)P) continue;
      const uint32_t at = s_base[p] + rank[e], place = threadIdx.x * kPer + e;
      const uint32_t chunk = s_first[p] + rank[e] / kFdByteChunk;
      if (rank[e] % kFdByteChunk == 0) {
        s_byte[at] = 1;
        atomicOr(&s_at[chunk], place);
        continue;
      }
      const uint32_t far = place - s_place[at - 1];
      s_byte[at] = (uint8_t)(far < 256u ? far : 0u);
      if (far >= 256u) atomicOr(&s_at[chunk], atomicCAS(&s_far[chunk], 0u, far) ? kFdFar | kFdSeveral : kFdFar);
    }
    __syncthreads();
    uint4 *row = reinterpret_cast<uint4 *>(static_cast<uint8_t *>(order) + (size_t)blockIdx.x * kFdByteRow);
    for (int i = threadIdx.x; i < kFdByteRow / 16; i += kFdBlock) row[i] = reinterpret_cast<const uint4 *>(s_byte)[i];
    if (threadIdx.x < kFdByteChunks)
      chunk_at[(size_t)blockIdx.x * kFdByteChunks + threadIdx.x] = s_at[threadIdx.x] | s_far[threadIdx.x] << 16;
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
// The lists of a group share the lines of the tables, so a group's workgroups belong on one die: the grid is as many groups
// wide as make a multiple of the eight dies that workgroups are dealt to in turn (268 M elements, sixteen lists, 147 groups:
// 18.5 us, with 152 12.5).  A tile's range of a list spans eight words there (22 us with one, 16 with five, and with eight 2 us more).
constexpr int kFdCountAhead = 5;
__global__ __launch_bounds__(kFdGroup) void k_fd_count(const uint32_t *__restrict__ below, uint32_t tiles, int P,
                                                       FdLists lists, uint32_t *__restrict__ vstart,
                                                       uint32_t *__restrict__ gsum, int32_t *status) {
  __shared__ uint32_t s_scan[kFdGroup / 64 + 1];
  const uint32_t tile = blockIdx.x * (uint32_t)kFdGroup + threadIdx.x;
  if (blockIdx.x * (uint32_t)kFdGroup >= tiles) return;
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
// 132, 100 and 101, 64 195, 203 and 212.  (Up to sixteen lists come here beyond 1.88e9 elements only, fd_of_bytes: eight
// words would gain 2 to 4 % from 24 lists on and lose 6 to 54 % there.)
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

// 0.0f + v for a tile put together in LDS, and out with it in 16-byte pieces, consecutive threads consecutive pieces:
// every store instruction fills whole lines.  By the whole workgroup; fix: some of the values may need the sum.
template <typename S, int TILE, int BLOCK>
__device__ inline void fd_write_tile(const S *s_tile, uint32_t tile_base, uint32_t n, bool fix, S *__restrict__ dense) {
  if ((reinterpret_cast<uintptr_t>(dense) & 15u) == 0 && tile_base + (uint32_t)TILE <= n) {
    constexpr int kAll = (int)(TILE * sizeof(S) / 16);
    constexpr int kPieces = (kAll + BLOCK - 1) / BLOCK;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(s_tile);
    u32x4 *dst = reinterpret_cast<u32x4 *>(dense + tile_base);
    u32x4 piece[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int at = i * BLOCK + (int)threadIdx.x;
      piece[i] = src[(i + 1) * BLOCK <= kAll || at < kAll ? at : 0];
    }
    if (fix) fd_values(piece, S(0));
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int at = i * BLOCK + (int)threadIdx.x;
      if ((i + 1) * BLOCK <= kAll || at < kAll) __builtin_nontemporal_store(piece[i], dst + at);
    }
  } else {
    for (uint32_t e = threadIdx.x; e < (uint32_t)TILE && tile_base + e < n; e += BLOCK)
      dense[tile_base + e] = fd_value<S>(s_tile[e]);
  }
}

template <typename S, int TILE, int BLOCK>
__device__ inline void fd_clear_tile(S *s_tile) {
  uint4 *z = reinterpret_cast<uint4 *>(s_tile);
#pragma unroll
  for (int i = 0; i * BLOCK < (int)(TILE * sizeof(S) / 16); ++i) {
    const int at = i * BLOCK + (int)threadIdx.x;
    if ((i + 1) * BLOCK <= (int)(TILE * sizeof(S) / 16) || at < (int)(TILE * sizeof(S) / 16)) z[at] = make_uint4(0, 0, 0, 0);
  }
}

// One workgroup per tile.  Lane p of every wave knows list p's members in the tile, the first bit of their range
// and where its values start; the lists' members are cut into chunks of 576, dealt to the waves in turn.  A
// wave gets the chunk's bits as nine 64-bit words in scalar registers: the word is the mask of the lanes whose
// member has a value, a lane's value is the one numbered by the set bits below it, and its place in the tile is
// the chunk's next entry of the dictionary, so that all loads are consecutive, nine of each kind in flight.  The
// places written are put together in LDS and leave with full-width stores.
// For 17 to 64 lists, and fewer beyond 1.88e9 elements.  Bound by the work per chunk, of which more lists make more and
// emptier ones: a decode of 134 M bf16 elements, 10 % set, takes 140 us with 17 lists (0.58 GB, 4.1 TB/s), 166 with 24, 201
// with 32, 334 with 64; 67 M fp32 99, 113, 132 and 198.  The figures below are from the time when sixteen lists came here
// too: 62 M bf16 elements, 71 % set, and 268 M, 11 % set (1.13 GB; 241 us in the end).
// What a 64th of a chunk costs beside its loads counts: places read without a look at the end of the list (the
// dictionary goes on behind it), values clamped only where they end, and 0.0f + v taken for what is written out as a
// whole instead of each value: 268 M 260 -> 249 us; chunks of nine words instead of ten, of which two were past most
// lists' ends, 241.  Slower: the bits by scalar loads (289; nine cache lines one after the other), the low bytes of the
// places alone with the high ones counted from where they wrap (0.86 GB, 275: seven instructions more per word).
// One SET bit per thread and turn, looked up in staged copies of the tile's bytes and values, took 307 us for the 62 M
// and 411 for the 268 M; with each value's load in a branch of its own, which makes the compiler wait for it there,
// this kernel took 129 and 428 (79 and 300 without).
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
  fd_clear_tile<S, kFdTile, kBlock>(s_tile);
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
  fd_write_tile<S, kFdTile, kBlock>(s_tile, tile_base, n, true, dense);
  if (odd && lane == 0) atomicOr(status, ZEN_STAT_BAD_INDEX);
}

// The kernel for dictionaries of bytes.  A wave takes a chunk of a list's members, a lane eight of them: their distances
// are one 8-byte load, their bits of the bitmap two bytes, and one prefix sum across the lanes gives every lane both the
// place in front of its first member and the number of its first value.  The lanes list the places of their members that
// have a value, in LDS, and the values go there with consecutive lanes on consecutive values.
// Bound by the three trips to memory of a tile, one after the other (743 M bf16 elements, sixteen lists, 6 % set: the
// waves wait 60 % of their time), and by the vector instructions (475 a wave of a tile): 268 M bf16 elements, sixteen
// lists, 11 % set, are 0.91 GB and a decode of 203 us, 4.5 TB a second (with places of 16 bits 249 us and 1.17 GB);
// fd_of_bytes has more. Slower (figures from the kernel's first form, 209 us there): a lane that fetches the values of
// its own members (eight loads that touch the same lines; 268 M: 316); tiles of 7680 elements, whose lists of 480
// members go beyond a chunk in one case of fifteen, and one of a tile's four waves takes five chunks where the others
// take four; 512 threads (40 more); four chunks of a wave under way together, all their loads in front (registers: 209
// at six waves a SIMD, 20 more at eight).
template <typename S>
__global__ __launch_bounds__(fd_tile_block<S>(), 8) void k_fd_tiles_bytes(
    const uint8_t *__restrict__ order, const uint32_t *__restrict__ chunk_at, const uint32_t *__restrict__ below,
    const uint32_t *__restrict__ vstart, const uint32_t *__restrict__ gpre, int P, FdDivisor n, FdDivisor npp, FdLists lists,
    S *__restrict__ dense, int32_t *status) {
  constexpr int kBlock = fd_tile_block<S>();
  __shared__ __attribute__((aligned(16))) S s_tile[kFdByteTile];
  __shared__ uint16_t s_list[kBlock / 64][kFdByteChunk];
  __shared__ uint32_t s_special;  // a value that 0.0f + v changes: -0 or a NaN
  const uint32_t tile = blockIdx.x;
  const uint32_t tile_base = tile * (uint32_t)kFdByteTile;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  uint32_t b0 = 0, b1 = 0, v0 = 0;
  if (lane < P) {
    const size_t at = (size_t)tile * P + lane;
    b0 = below[at];
    b1 = below[at + P];
    v0 = vstart[at] + gpre[(size_t)(tile / kFdGroup) * P + lane];
  }
  const uint32_t starts = lane < kFdByteChunks ? chunk_at[(size_t)tile * kFdByteChunks + lane] : 0u;
  fd_clear_tile<S, kFdByteTile, kBlock>(s_tile);
  if (threadIdx.x == 0) s_special = 0;
  uint32_t cnt = b1 - b0;
  if (cnt > (uint32_t)kFdByteTile) cnt = 0;  // cannot be with a table this library built
  const uint32_t room = (cnt + kFdLane - 1) / kFdLane * kFdLane, chunks = (cnt + kFdByteChunk - 1) / kFdByteChunk;
  const uint32_t incl = wave_inclusive_scan(room), cincl = wave_inclusive_scan(chunks);
  const uint32_t nchunks = (uint32_t)__builtin_amdgcn_readlane((int)cincl, 63);
  const bool odd = __builtin_amdgcn_readlane((int)incl, 63) > kFdByteRow || nchunks > (uint32_t)kFdByteChunks;  // cannot be either
  const uint8_t *row = order + (size_t)tile * kFdByteRow;
  uint16_t *list = s_list[wave];
  __syncthreads();
  // What a chunk asks memory for: its distances, and for every lane the byte of the bitmap that holds its first bit and
  // the one behind that.  The next chunk's are asked for while this one's are worked on.
  // (so are the list's pointers and lengths: a wave would wait for the constants' cache in front of every use)
  struct Asked {
    int p;
    uint32_t j0, bytes, have;
    const uint8_t *bitmap;
    const char *val;
    uint8_t lo, hi;
    u32x2 far;
  };
  auto ask = [&](uint32_t c) {
    Asked a;
    a.p = (int)__popcll(__ballot(cincl <= c));  // the chunk's list
    a.j0 = (c - (uint32_t)__builtin_amdgcn_readlane((int)(cincl - chunks), a.p)) * kFdByteChunk;
    // (past the members: the next list's distances, or what follows the last)
    a.far = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(
        row + (uint32_t)__builtin_amdgcn_readlane((int)(incl - room), a.p) + a.j0 + lane * kFdLane));
    a.bytes = lists.bytes[a.p];
    a.bitmap = lists.bitmap[a.p];  // of a list without one: readable all the same
    a.have = lists.vals[a.p];
    a.val = static_cast<const char *>(lists.val[a.p]);
    const uint32_t last = a.bytes ? a.bytes - 1u : 0u;
    const uint32_t at = (((uint32_t)__builtin_amdgcn_readlane((int)b0, a.p) + a.j0) >> 3) + (uint32_t)lane;
    const uint32_t at0 = at < last ? at : last, at1 = at + 1u < last ? at + 1u : last;
    a.lo = a.bitmap[at0];
    a.hi = a.bitmap[at1];
    return a;
  };
  // Places are sums of the dictionary's distances, and the dictionary is the caller's memory: one that this library did not
  // build for these sizes must not reach beyond the tile in LDS.  (134 M bf16 elements, sixteen lists, 10 % set: 117 us
  // with and without.)
  uint32_t last_place = 0;
  auto put_one = [&](uint32_t place, S v) {
    last_place = last_place > place ? last_place : place;
    s_tile[place < (uint32_t)kFdByteTile ? place : 0u] = v;
  };
  Asked next{};
  if ((uint32_t)wave < nchunks && !odd) next = ask((uint32_t)wave);
#pragma unroll 1
  for (uint32_t c = (uint32_t)wave; c < nchunks && !odd; c += kBlock / 64) {
    const Asked now = next;
    next = ask(c + kBlock / 64 < nchunks ? c + kBlock / 64 : c);
    const int p = now.p;
    const uint32_t j0 = now.j0;
    const u32x2 far = now.far;
    const uint32_t members = (uint32_t)__builtin_amdgcn_readlane((int)cnt, p) - j0;  // from here on, > 0
    const uint32_t bit0 = (uint32_t)__builtin_amdgcn_readlane((int)b0, p) + j0;
    const uint32_t start = (uint32_t)__builtin_amdgcn_readlane((int)starts, (int)c);
    // the members' bits; those past the members and past the bitmap's end are zero
    const uint32_t before = (uint32_t)lane * kFdLane;
    uint32_t bits;
    {
      const uint32_t limit = now.bytes * 8u;
      const uint32_t has = bit0 < limit ? limit - bit0 : 0u;  // bits the bitmap has from the chunk's first on
      const uint32_t end = has < members ? has : members;
      const uint32_t left = end > before ? end - before : 0u;
      bits = __builtin_amdgcn_ubfe((uint32_t)now.lo | (uint32_t)now.hi << 8, bit0 & 7u, left < (uint32_t)kFdLane ? left : (uint32_t)kFdLane);
    }
    // set bits of the tile's range in front of the chunk: the list's earlier chunks in this tile
    uint32_t nth = (uint32_t)__builtin_amdgcn_readlane((int)v0, p);
    if (j0) {  // 128 bits per lane
      const uint32_t from = bit0 - j0 + (uint32_t)lane * (kFdTile / 64);
      const uint32_t to = from + kFdTile / 64;
      nth += wave_sum(from < bit0 ? popcount_range<1>(now.bitmap, now.bytes, from, to < bit0 ? to : bit0) : 0u);
    }
    nth = (uint32_t)__builtin_amdgcn_readfirstlane((int)nth);
    // Both prefix sums in one word: places (below 2^14; those of lanes past the members stay below 2^18) in the low 18 bits,
    // values above.
    const uint32_t mine = __builtin_amdgcn_sad_u8(far.x, 0u, __builtin_amdgcn_sad_u8(far.y, 0u, (uint32_t)__popc(bits) << 18));
    const uint32_t all = wave_inclusive_scan(mine);
    uint32_t set = (uint32_t)__builtin_amdgcn_readlane((int)all, 63) >> 18;
    const uint32_t k = (all - mine) >> 18;
    const uint32_t have = now.have;
    if (nth + set > have) {  // more set bits than values: the missing ones count as unset
      set = have > nth ? have - nth : 0u;
      while (bits && k + (uint32_t)__popc(bits) > set) bits &= ~(0x80000000u >> __clz((int)bits));
    }
    if (set == 0) continue;
    const char *val = now.val + (size_t)nth * sizeof(S);
    if (start & kFdSeveral) {  // several distances that do not fit their bytes: whose the places are is hashed out
      uint32_t seen = 0;
      for (uint32_t t0 = 0; t0 < (uint32_t)kFdByteTile; t0 += 64) {
        const uint32_t t = t0 + (uint32_t)lane;
        const bool member = tile_base + t < n.d && part_of(tile_base + t, n, npp) == (uint32_t)p;
        const unsigned long long who = __ballot(member);
        const uint32_t j = seen + __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u)) - j0;
        seen += (uint32_t)__popcll(who);
        const uint32_t theirs = (uint32_t)__shfl((int)bits, (int)(j / kFdLane) & 63, 64);
        const uint32_t front = (uint32_t)__shfl((int)k, (int)(j / kFdLane) & 63, 64);
        const uint32_t bit = j % kFdLane;
        if (member && j < (uint32_t)kFdByteChunk && ((theirs >> bit) & 1u))
          s_special = 1, s_tile[t] = reinterpret_cast<const S *>(val)[front + (uint32_t)__popc(theirs & ((1u << bit) - 1u))];
      }
      continue;
    }
    // One that does not fit, of the member whose byte is zero: its lane adds the distance to the places that it has listed
    // from there on, the lanes behind it begin that much further.  (Hashed out like several, one such chunk of a call cost
    // 15 to 20 us where it came late: sixteen lists, 141 040 elements 35 us and 16 so, 16.8 M fp32 55 and 35, 134 M bf16
    // with eight of them 118 and 107.)
    auto far_member = [&] {  // kFdLane: none of this lane's
      const uint32_t zx = (far.x - 0x01010101u) & ~far.x & 0x80808080u, zy = (far.y - 0x01010101u) & ~far.y & 0x80808080u;
      const uint32_t i = zx ? (uint32_t)__ffs((int)zx) / 8u - 1u : zy ? (uint32_t)__ffs((int)zy) / 8u + 3u : (uint32_t)kFdLane;
      return before + i < members ? i : (uint32_t)kFdLane;
    };
    uint32_t front = (start & kFdPlace) + ((all - mine) & 0x3ffffu) - 1u;
    if (start & kFdFar) {
      const int who = __ffsll(__ballot(far_member() < (uint32_t)kFdLane));  // and one
      if (who && lane >= who) front += start >> 16;
    }
    // The places of those that have a value are listed in its order, and the values go there with consecutive lanes on
    // consecutive values: a lane that fetches its own members' reads the same lines as its neighbours eight times over.
    auto put = [&](auto rows) {
      constexpr int kRows = decltype(rows)::value;
      S v[kRows];
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        const uint32_t at = (uint32_t)(i * 64 + lane);
        v[i] = *reinterpret_cast<const S *>(val + (uint32_t)((at < set ? at : set - 1u) * sizeof(S)));
      }
      uint32_t place = front;
      int mark = (int)__brev(bits);
      uint16_t *to = list + k;
#pragma unroll
      for (int i = 0; i < kFdLane; ++i) {
        place += ((i < 4 ? far.x : far.y) >> (8 * (i & 3))) & 0xffu;
        if (mark < 0) *to++ = (uint16_t)place;
        mark <<= 1;
      }
      if (kRows == kFdLane && (start & kFdFar)) {
        const uint32_t i = far_member();
        if (i < (uint32_t)kFdLane)
          for (uint16_t *e = list + k + (uint32_t)__popc(bits & ((1u << i) - 1u)); e < to; ++e) *e = (uint16_t)(*e + (start >> 16));
      }
      __builtin_amdgcn_wave_barrier();
      bool special = false;
#pragma unroll
      for (int i = 0; i < kRows; ++i) special |= __builtin_amdgcn_classf(KeyOf<S>::to_f32(v[i]), 0x23);
      if (special) s_special = 1;
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        const uint32_t at = (uint32_t)(i * 64 + lane);
        if (at < set) put_one(list[at], v[i]);
      }
      __builtin_amdgcn_wave_barrier();
    };
    if (start & kFdFar)
      put(std::integral_constant<int, kFdLane>{});
    else if (set <= 64u)
      put(std::integral_constant<int, 1>{});
    else if (set <= 128u)
      put(std::integral_constant<int, 2>{});
    // (a quarter to half of a chunk set; by the eight rows of all those denser fp32 calls were slower than with places of
    // 16 bits: 67 M fp32, us, with 16 bits, eight rows, four: sixteen lists, 45 % set 94, 98 and 94; eight, 48 % 111, 116
    // and 114; four, 30 % 113, 118 and 116.  134 M bf16, sixteen lists, 45 %: 134, 124 and 118.)
    else if (set <= 256u)
      put(std::integral_constant<int, 4>{});
    else
      put(std::integral_constant<int, kFdLane>{});
  }
  __syncthreads();
  fd_write_tile<S, kFdByteTile, kBlock>(s_tile, tile_base, n.d, s_special != 0, dense);
  if ((odd && lane == 0) || last_place >= (uint32_t)kFdByteTile) atomicOr(status, ZEN_STAT_BAD_INDEX);
}

// Dictionaries of bytes (see kFdByteLists), as long as their tiles' groups have a thread each in k_fd_groups (1.88e9 elements).
// A decode with places of 16 bits and with bytes, us, 10 % and 70 % set.  134 M bf16: one list 167, 147 and 169, 164;
// two 175, 154 and 177, 172; three 163, 144 and 165, 161; four 172, 155 and 175, 173; eight 169, 150 and 172, 168;
// twelve 221, 192 and 224, 201; sixteen 132, 108 and 137, 129.  67 M fp32: one 117, 115 and 119, 124; two 116, 113 and
// 118, 123; three 111, 110 and 114, 119; four 113, 112 and 116, 121; eight 109, 108 and 113, 117; twelve 137, 130 and
// 139, 137; sixteen 89, 85 and 102, 102.  Up to 9 M elements bytes take 5 to 30 % less, and the dictionary is built in
// three quarters to six sevenths of the time.  (fp32 of few lists with most of their members set loses up to 5 %: a
// dictionary serves both types.)
inline bool fd_of_bytes(int64_t numel, int P) {
  return P <= kFdByteLists && ceil_div(numel, kFdByteTile) <= (int64_t)kFdGroupsMax * kFdGroup;
}
inline uint32_t fd_tiles(int64_t numel, int P) { return (uint32_t)ceil_div(numel, fd_of_bytes(numel, P) ? kFdByteTile : kFdTile); }
// (a chunk's places are read as if it were full)
inline size_t fd_order_bytes(int64_t numel, int P) {
  const size_t tiles = fd_tiles(numel, P);
  return align_up(fd_of_bytes(numel, P) ? tiles * kFdByteRow + kFdByteChunk : (tiles * kFdTile + kFdMembers) * sizeof(uint16_t), 256);
}
inline size_t fd_chunk_bytes(int64_t numel, int P) {
  return fd_of_bytes(numel, P) ? align_up((size_t)fd_tiles(numel, P) * kFdByteChunks * sizeof(uint32_t), 256) : 0;
}
inline size_t fd_table_bytes(int64_t numel, int P) { return align_up(((size_t)fd_tiles(numel, P) + 1) * P * sizeof(uint32_t), 256); }
inline size_t fd_vstart_bytes(int64_t numel, int P) { return align_up((size_t)fd_tiles(numel, P) * P * sizeof(uint32_t), 256); }
inline size_t fd_gsum_bytes(int64_t numel, int P) { return align_up((size_t)fd_groups(fd_tiles(numel, P)) * P * sizeof(uint32_t), 256); }

int fd_check(int64_t numel, int partitions) {
  if (numel <= 0 || numel > 0x7fffffffll || partitions < 1 || partitions > kFdMaxLists || numel / partitions == 0)
    return fail(ZEN_EINVAL, "zen_bitmap_dense: need 0 < partitions <= 64 and partitions <= numel < 2^31");
  return ZEN_OK;
}

template <typename S>
void fd_launch_tiles(const void *dict, const uint8_t *chunk_at, const uint32_t *below, const uint32_t *vstart,
                     const uint32_t *gsum, uint32_t tiles, int P, int64_t numel, const FdLists &lists, void *dense,
                     int32_t *status, hipStream_t s) {
  const dim3 grid(tiles), block(fd_tile_block<S>());
  if (fd_of_bytes(numel, P))
    k_fd_tiles_bytes<S><<<grid, block, 0, s>>>(static_cast<const uint8_t *>(dict), reinterpret_cast<const uint32_t *>(chunk_at),
                                               below, vstart, gsum, P, fd_divisor((uint32_t)numel), fd_divisor((uint32_t)(numel / P)), lists,
                                               static_cast<S *>(dense), status);
  else
    k_fd_tiles<S><<<grid, block, 0, s>>>(static_cast<const uint16_t *>(dict), below, vstart, gsum, P, (uint32_t)numel, lists,
                                         static_cast<S *>(dense), status);
}

}  // namespace
}  // namespace zen

extern "C" {

size_t zen_bitmap_dense_dict_bytes(int64_t numel, int partitions) {
  if (zen::fd_check(numel, partitions) != ZEN_OK) return 0;
  return zen::fd_order_bytes(numel, partitions) + zen::fd_chunk_bytes(numel, partitions) + zen::fd_table_bytes(numel, partitions);
}

int zen_bitmap_dense_dict(int64_t numel, int partitions, void *dict, int64_t *members, void *stream) {
  using namespace zen;
  const int rc = fd_check(numel, partitions);
  if (rc != ZEN_OK) return rc;
  if (!dict || (reinterpret_cast<uintptr_t>(dict) & 15u)) return fail(ZEN_EINVAL, "zen_bitmap_dense_dict: null or unaligned dictionary");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool of_bytes = fd_of_bytes(numel, partitions);
  uint8_t *chunk_at = static_cast<uint8_t *>(dict) + fd_order_bytes(numel, partitions);
  uint32_t *below = reinterpret_cast<uint32_t *>(chunk_at + fd_chunk_bytes(numel, partitions));
  const uint32_t tiles = fd_tiles(numel, partitions);
  const size_t lds = (size_t)partitions * (kFdBlock + kFdChunkRow) * sizeof(uint16_t) + (of_bytes ? kFdByteRow * 3u : 0u);
  const auto fill = of_bytes ? k_fd_order<true> : k_fd_order<false>;
  if (lds > 32768)  // beyond what a launch may ask for without saying so first
    ZEN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(fill), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  fill<<<dim3(tiles), dim3(kFdBlock), lds, s>>>(fd_divisor((uint32_t)numel), fd_divisor((uint32_t)(numel / partitions)), partitions, dict,
                                                reinterpret_cast<uint32_t *>(chunk_at), below);
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
    lists.bitmap[p] = bitmap_bytes[p] ? bitmaps[p] : static_cast<const uint8_t *>(dict);
    lists.bytes[p] = (uint32_t)(bitmap_bytes[p] < (1ll << 28) ? bitmap_bytes[p] : 1ll << 28);
    lists.val[p] = values[p];
    lists.vals[p] = (uint32_t)(value_count[p] < (1ll << 31) ? value_count[p] : 1ll << 31);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint8_t *chunk_at = static_cast<const uint8_t *>(dict) + fd_order_bytes(numel, partitions);
  const uint32_t *below = reinterpret_cast<const uint32_t *>(chunk_at + fd_chunk_bytes(numel, partitions));
  uint32_t *vstart = static_cast<uint32_t *>(workspace);
  uint32_t *gsum = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(workspace) + fd_vstart_bytes(numel, partitions));
  const uint32_t tiles = fd_tiles(numel, partitions);
  const uint32_t groups = fd_groups(tiles);
  ProfScope prof(kProfDecodeFused, s);
  k_fd_count<<<dim3((groups + 7u) / 8u * 8u, (unsigned)partitions), dim3(kFdGroup), 0, s>>>(below, tiles, partitions, lists, vstart, gsum,
                                                                       status);
  ZEN_LAUNCH_CHECK("k_fd_count");
  k_fd_groups<<<dim3((unsigned)partitions), dim3(kFdGroupsMax), 0, s>>>(gsum, groups, partitions, lists, status);
  ZEN_LAUNCH_CHECK("k_fd_groups");
  if (dtype == ZEN_BF16)
    fd_launch_tiles<uint16_t>(dict, chunk_at, below, vstart, gsum, tiles, partitions, numel, lists, dense, status, s);
  else
    fd_launch_tiles<uint32_t>(dict, chunk_at, below, vstart, gsum, tiles, partitions, numel, lists, dense, status, s);
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
