// The threshold compress() applies (train.py:75-84): the k-th largest magnitude of a gathered sample.
//
// The sample is 1 % of a gradient bucket, at random places: what the call cannot do without is one memory line
// per sample element.  A radix select behind a gather took 6 to 8 dependent launches, each a few microseconds of
// work; here the histogram is taken while the elements arrive, at 15 bits of the magnitude (for bf16 the whole
// key), so that one more workgroup finds the k-th:
//   up to kOneMax elements    one workgroup does everything in one launch, the elements in registers;
//   more, bf16                k_sample_count (every workgroup keeps 32768 16-bit counters in LDS and writes them
//                             out, with sums of 64 neighbours each: nothing has to be zero beforehand and no
//                             atomic leaves the compute unit), k_sample_pick (one workgroup);
//   more, fp32                the elements are kept too, and the low halves of those in the k-th's bin decide: in the
//                             picking workgroup up to 16 384 elements, else a third kernel lists them and its last
//                             workgroup picks among them.
#include "zen_select.h"

namespace zen {
namespace {

constexpr int kBins = 32768;       // 15 bits of the magnitude key
constexpr int kBlock = 1024;
// One workgroup as long as that is no slower than the two launches for larger samples: every 1024 elements cost it
// up to a microsecond, the gather of a single compute unit and its counting loop, and the other way costs a launch of the
// host's.  A call on either side of the line, us by events: bf16 4096 elements 12.8, 5120 13.5, 5121 (two launches) 14.3,
// 8192 14.4; fp32 4096 15.8, 5120 16.8, 5121 16.1, 8192 16.4.  In front of a compress and a load balance, which are bound by
// the host, one launch stays ahead a little longer: 4565 bf16 elements 100 and 104.5 us a pass, 4000 fp32 102.5 and 105, but
// 7000 bf16 106 and 103.
constexpr int kOneItems = 5;
constexpr int64_t kOneMax = kOneItems * kBlock;
constexpr int kGroup = 64;         // bins per sum
constexpr int kGroups = kBins / kGroup;
// elements per thread up to which the picking workgroup looks at an fp32 sample's low halves itself (a call for 10 486
// elements 20.4 us with the third launch, 17.1 without; 32 registers for them 18.1, and 20.0 instead of 22.0 at 32 768)
constexpr int kFewItems = 16;
constexpr int kRound = 4;          // elements per thread in flight in the counting kernel
constexpr int64_t kShare = 65535;  // elements a workgroup counts at most (16-bit counters)
// the bins' 16-bit counters, two to a word, one word of padding per 32 (a thread reads 16 neighbouring words)
constexpr int kHistWords = kBins / 2 + kBins / 64;
__device__ inline int hist_word(int w) { return w + (w >> 5); }

// Adds one to the counter of every lane's bin (lanes without `live` add nothing).  The lanes that share the
// first live lane's bin add together: in a mostly zero gradient nearly every element meets in one bin, and a
// wave's adds to one address are carried out one after the other.
__device__ inline void count_bin(uint32_t *hist, uint32_t bin, bool live) {
  const uint64_t all = __ballot(live);
  if (!all) return;
  const int lead = __ffsll((unsigned long long)all) - 1;
  const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)bin, lead);
  const uint64_t same = __ballot(live && bin == first);
  const bool with_first = live && bin == first;
  const uint32_t n = with_first ? (uint32_t)__popcll(same) : 1u;
  if (live && (!with_first || lane_id() == lead)) atomicAdd(&hist[hist_word((int)(bin >> 1))], n << (16 * (bin & 1u)));
}

struct Pick {
  uint32_t bin, above, count;  // the bin that holds the rank-th largest, elements in the bins above it and in it
};

// The bin of the histogram in LDS that holds the rank-th largest (1 <= rank <= elements counted).  By the whole
// workgroup; smem: kBlock / 64 + 1 words; *out is valid behind the barrier at the end.
__device__ inline void pick_bin(const uint32_t *hist, uint32_t rank, uint32_t *smem, Pick *out) {
  constexpr int kWords = kBins / 2 / kBlock;
  uint32_t c[kWords];
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < kWords; ++j) {  // from the top down
    c[j] = hist[hist_word(kBins / 2 - 1 - (int)(threadIdx.x * kWords + j))];
    mine += (c[j] & 0xffffu) + (c[j] >> 16);
  }
  uint32_t total;
  uint32_t above = block_exclusive_scan<uint32_t, kBlock>(mine, smem, &total);
  if (above < rank && rank <= above + mine) {
#pragma unroll
    for (int j = 0; j < kWords; ++j) {
#pragma unroll
      for (int h = 1; h >= 0; --h) {
        const uint32_t n = h ? c[j] >> 16 : c[j] & 0xffffu;
        if (above < rank && rank <= above + n) {
          out->bin = 2u * (uint32_t)(kBins / 2 - 1 - (int)(threadIdx.x * kWords + j)) + (uint32_t)h;
          out->above = above;
          out->count = n;
        }
        above += n;
      }
    }
  }
  __syncthreads();
}

__device__ inline void clear_hist(uint32_t *hist) {
  for (int i = threadIdx.x; i < kHistWords; i += kBlock) hist[i] = 0;
}

// Positions at[first + i * kBlock], i < ITEMS, of the sample (those at or past `end` and those outside the tensor
// read element 0 as zero; the latter are flagged): all loads of a round in flight together.
template <typename S, int ITEMS>
__device__ inline void gather(const S *__restrict__ in, int64_t n, const int64_t *__restrict__ at, int64_t first,
                              int64_t end, S (&v)[ITEMS], int32_t *status) {
  int64_t pos[ITEMS];
  bool bad = false;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int64_t j = first + (int64_t)i * kBlock;
    pos[i] = at ? __builtin_nontemporal_load(at + (j < end ? j : end - 1)) : (j < end ? j : end - 1);
    if (pos[i] < 0 || pos[i] >= n) {
      bad = true;
      pos[i] = -1;
    }
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) v[i] = __builtin_nontemporal_load(in + (pos[i] >= 0 ? pos[i] : 0));
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    if (pos[i] < 0) v[i] = 0;
  if (bad) atomicOr(status, ZEN_STAT_BAD_INDEX);
}

// Everything in one workgroup.  Bound by the chain gather - histogram - search: 5 us for 93 bf16 elements (six
// launches before: 26 us a call, now 12).
template <typename S>
__global__ __launch_bounds__(kBlock) void k_sample_one(const S *__restrict__ in, int64_t n,
                                                       const int64_t *__restrict__ at, uint32_t s, uint32_t k,
                                                       uint32_t *__restrict__ thr, int32_t *status) {
  __shared__ uint32_t hist[kHistWords];
  __shared__ uint32_t smem[kBlock / 64 + 1];
  __shared__ Pick pick;
  __shared__ uint32_t low[2];
  clear_hist(hist);
  if (threadIdx.x < 2) low[threadIdx.x] = 0;
  constexpr int kItems = kOneItems;
  S v[kItems];
  gather<S, kItems>(in, n, at, threadIdx.x, s, v, status);
#pragma unroll
  for (int i = 0; i < kItems; ++i) v[i] &= (S)KeyOf<S>::kMask;
  __syncthreads();
  constexpr int kShift = KeyOf<S>::kBits - 15;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    count_bin(hist, (uint32_t)v[i] >> kShift, threadIdx.x + (uint32_t)i * kBlock < s);
  }
  __syncthreads();
  pick_bin(hist, k, smem, &pick);
  const uint32_t top = pick.bin;
  if (sizeof(S) == 2) {
    if (threadIdx.x == 0) {
      thr[0] = top;
      thr[1] = pick.above + pick.count;
    }
    return;
  }
  // fp32: 15 of the 16 bits that are left, then the last
  const uint32_t above = pick.above;
  __syncthreads();
  clear_hist(hist);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const uint32_t key = (uint32_t)v[i];
    count_bin(hist, (key & 0xffffu) >> 1, threadIdx.x + (uint32_t)i * kBlock < s && (key >> 16) == top);
  }
  __syncthreads();
  pick_bin(hist, k - above, smem, &pick);
  const uint32_t high = (top << 15) | pick.bin;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const uint32_t key = (uint32_t)v[i];
    const bool live = threadIdx.x + (uint32_t)i * kBlock < s && (key >> 1) == high;
    const uint64_t odd = __ballot(live && (key & 1u)), all = __ballot(live);
    if (all && lane_id() == 0) {
      atomicAdd(&low[1], (uint32_t)__popcll(odd));
      atomicAdd(&low[0], (uint32_t)__popcll(all & ~odd));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t over = above + pick.above, odd = low[1];
    const uint32_t bit = over + odd >= k ? 1u : 0u;
    thr[0] = (high << 1) | bit;
    thr[1] = over + odd + (bit ? 0u : low[0]);
  }
}

struct SampleTables {
  uint16_t *sums;    // [workgroups][kGroups] per workgroup: elements in 64 neighbouring bins
  uint16_t *bins;    // [workgroups][kBins]
  uint32_t *sample;  // fp32: the magnitude keys
  uint16_t *members; // fp32: low halves of the keys in the k-th's bin
  uint32_t *state;   // fp32: [0] bin, [1] rank inside it, [2] elements above it, [3] members listed, [4] workgroups done
};

// Bound by the sample's lines: 2.7 M elements of a 537 MB tensor at random places are 344 MB of them, which come at 51 a
// nanosecond at most, 53 us.  The gather's loads are streamed (nontemporal): of a line one element is wanted, and a tensor of
// gigabytes would only push others out (with the tensor cold in every cache a call 72 us, 120 with plain loads).  Trips to
// memory overlap: the first places are asked for in front of the clearing of the counters, a round's elements in front of the
// counting of the round before, their places a round earlier still; and of the counters only groups that hold something are
// written out, 64 KB a workgroup else.  One after the other and all written: 2.7 M bf16 elements 62.5 us, so 57.3; 620 000
// 21.8 and 17.2; 129 000 fp32 11.9 and 7.4; 10 486 8.2 and 4.9.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_sample_count(const S *__restrict__ in, int64_t n,
                                                         const int64_t *__restrict__ at, int64_t s, int64_t share,
                                                         SampleTables tb, int32_t *status) {
  __shared__ uint32_t hist[kHistWords];
  constexpr int kShift = KeyOf<S>::kBits - 15;
  constexpr int64_t kStep = (int64_t)kRound * kBlock;
  const int64_t begin = (int64_t)blockIdx.x * share;
  const int64_t end = begin + share < s ? begin + share : s;
  int64_t pos[2][kRound];
  S v[2][kRound];
  uint32_t wrong[2], any = 0;  // bit i: element i's place is outside the tensor (element 0 is read, as zero)
  auto ask_places = [&](int64_t j0, int64_t (&p)[kRound]) {
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      const int64_t j = j0 + threadIdx.x + (int64_t)i * kBlock;
      p[i] = at ? __builtin_nontemporal_load(at + (j < end ? j : end - 1)) : (j < end ? j : end - 1);
    }
  };
  auto ask_elements = [&](const int64_t (&p)[kRound], S (&e)[kRound], uint32_t &out) {
    out = 0;
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      const bool in_range = (uint64_t)p[i] < (uint64_t)n;
      out |= in_range ? 0u : 1u << i;
      e[i] = __builtin_nontemporal_load(in + (in_range ? p[i] : 0));
    }
    any |= out;
  };
  auto count = [&](int64_t j0, const S (&e)[kRound], uint32_t out) {
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      const int64_t j = j0 + threadIdx.x + (int64_t)i * kBlock;
      const uint32_t key = out & (1u << i) ? 0u : e[i] & KeyOf<S>::kMask;
      count_bin(hist, key >> kShift, j < end);
      if (sizeof(S) == 4 && j < end) tb.sample[j] = key;
    }
  };
  ask_places(begin, pos[0]);
  if (begin + kStep < end) ask_places(begin + kStep, pos[1]);
  clear_hist(hist);
  ask_elements(pos[0], v[0], wrong[0]);
  __syncthreads();
  int64_t j0 = begin;
  // a round's elements are asked for in front of the counting of the one before, its places a round earlier still
  for (; j0 + kStep < end; j0 += 2 * kStep) {
    ask_places(j0 + 2 * kStep, pos[0]);  // (past the end: the last place once more)
    ask_elements(pos[1], v[1], wrong[1]);
    count(j0, v[0], wrong[0]);
    ask_places(j0 + 3 * kStep, pos[1]);
    ask_elements(pos[0], v[0], wrong[0]);
    count(j0 + kStep, v[1], wrong[1]);
  }
  if (j0 < end) count(j0, v[0], wrong[0]);
  if (any) atomicOr(status, ZEN_STAT_BAD_INDEX);
  __syncthreads();
  // thread t: 16 words = 32 bins, half a group
  uint32_t w[16];
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    w[j] = hist[hist_word((int)threadIdx.x * 16 + j)];
    sum += (w[j] & 0xffffu) + (w[j] >> 16);
  }
  sum += __shfl_xor(sum, 1, 64);
  if (sum) {  // (nobody looks at the bins of a group without elements)
    uint4 *bins = reinterpret_cast<uint4 *>(tb.bins + (size_t)blockIdx.x * kBins);
#pragma unroll
    for (int j = 0; j < 4; ++j) bins[threadIdx.x * 4 + j] = make_uint4(w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]);
  }
  if ((threadIdx.x & 1u) == 0) tb.sums[(size_t)blockIdx.x * kGroups + threadIdx.x / 2] = (uint16_t)sum;
}

// Sums of 16-bit counters over the workgroups of the counting kernel: COUNTERS of them, WORDS * 2 to a thread's load, by
// rows of threads side by side, BATCH rows of a thread in flight together.  acc: [COUNTERS] words of LDS, zeroed here.  A row
// counts where counted(row) says so.  (The rows that were left over from batches of eight were read one trip to memory after
// the other: k_sample_pick with 152 rows 6.5 us, 256 rows 8.7.)
template <int COUNTERS, int WORDS, int BATCH, typename Counted>
__device__ inline void sum_columns(const uint16_t *from, size_t stride, uint32_t rows, uint32_t *acc, Counted counted) {
  using Words = uint32_t __attribute__((ext_vector_type(WORDS)));
  constexpr uint32_t kColumns = COUNTERS / (2 * WORDS), kRows = kBlock / kColumns;
  for (int i = threadIdx.x; i < COUNTERS; i += kBlock) acc[i] = 0;
  __syncthreads();
  const uint32_t col = threadIdx.x % kColumns, row = threadIdx.x / kColumns;
  uint32_t c[2 * WORDS];
#pragma unroll
  for (int e = 0; e < 2 * WORDS; ++e) c[e] = 0;
#pragma unroll 1
  for (uint32_t r0 = row; r0 < rows; r0 += BATCH * kRows) {
    Words q[BATCH];
    bool in[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const uint32_t r = r0 + i * kRows < rows ? r0 + i * kRows : row;
      q[i] = *reinterpret_cast<const Words *>(from + (size_t)r * stride + col * 2 * WORDS);
      in[i] = counted(r) && r0 + i * kRows < rows;
    }
#pragma unroll
    for (int i = 0; i < BATCH; ++i)
#pragma unroll
      for (int e = 0; e < WORDS; ++e) {
        const uint32_t x = in[i] ? q[i][e] : 0u;
        c[2 * e] += x & 0xffffu;
        c[2 * e + 1] += x >> 16;
      }
  }
#pragma unroll
  for (int e = 0; e < 2 * WORDS; ++e)
    if (c[e]) atomicAdd(&acc[col * 2 * WORDS + e], c[e]);  // (most of a sample's bins are empty)
  __syncthreads();
}

// fp32: the threshold among the m elements in the k-th's bin `top`, by their low halves at(0..m), eight bits at a time;
// rank: the k-th's inside the bin, above: elements in the bins above it.  By the whole workgroup.
template <typename At>
__device__ inline void low_halves(uint32_t m, uint32_t top, uint32_t rank, uint32_t above, uint32_t *__restrict__ thr, At at) {
  __shared__ uint32_t hist[256];
  __shared__ uint32_t smem[kBlock / 64 + 1];
  __shared__ uint32_t found[3];
  uint32_t prefix = 0;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    if (threadIdx.x < 256) hist[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t rounds = (m + kBlock - 1) / kBlock;
    for (uint32_t r = 0; r < rounds; ++r) {
      const uint32_t j = r * kBlock + threadIdx.x;
      const uint32_t x = j < m ? at(j) : 0u;
      const bool live = j < m && (pass == 0 || (x >> 8) == prefix);
      const uint32_t digit = pass == 0 ? x >> 8 : x & 0xffu;
      const uint64_t all = __ballot(live);  // equal digits add together where they are all equal (see count_bin)
      if (all) {
        const int lead = __ffsll((unsigned long long)all) - 1;
        const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)digit, lead);
        if (__ballot(live && digit == first) == all) {
          if (lane_id() == lead) atomicAdd(&hist[first], (uint32_t)__popcll(all));
        } else if (live) {
          atomicAdd(&hist[digit], 1u);
        }
      }
    }
    __syncthreads();
    const uint32_t c = threadIdx.x < 256 ? hist[255 - threadIdx.x] : 0u;
    uint32_t total;
    const uint32_t before = block_exclusive_scan<uint32_t, kBlock>(c, smem, &total);
    if (before < rank && rank <= before + c) {
      found[0] = 255u - threadIdx.x;
      found[1] = before;
      found[2] = c;
    }
    __syncthreads();
    prefix = (prefix << 8) | found[0];
    rank -= found[1];
    above += found[1];
  }
  if (threadIdx.x == 0) {
    thr[0] = (top << 16) | prefix;
    thr[1] = above + found[2];
  }
}

// FEW (fp32): the sample's keys are few enough for this workgroup's registers, and it finishes the search itself.
template <typename S, bool FEW>
__global__ __launch_bounds__(kBlock) void k_sample_pick(SampleTables tb, uint32_t rows, uint32_t s, uint32_t k,
                                                        uint32_t *__restrict__ thr) {
  constexpr int kItems = FEW ? kFewItems : 1;
  uint32_t key[kItems];
  if (FEW) {  // on their way while the bin is found
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const uint32_t j = threadIdx.x + (uint32_t)i * kBlock;
      key[i] = tb.sample[j < s ? j : 0u];
    }
  }
  __shared__ uint32_t acc[kGroups];
  __shared__ uint32_t smem[kBlock / 64 + 1];
  __shared__ uint32_t found[3];
  sum_columns<kGroups, 4, FEW ? 1 : 8>(tb.sums, kGroups, rows, acc, [](uint32_t) { return true; });
  {
    const uint32_t c = threadIdx.x < kGroups ? acc[kGroups - 1 - threadIdx.x] : 0u;
    uint32_t total;
    const uint32_t above = block_exclusive_scan<uint32_t, kBlock>(c, smem, &total);
    if (above < k && k <= above + c) {
      found[0] = (uint32_t)(kGroups - 1) - threadIdx.x;
      found[1] = above;
    }
  }
  __syncthreads();
  const uint32_t group = found[0], over = found[1];
  sum_columns<kGroup, 2, FEW ? 1 : 4>(tb.bins + (size_t)group * kGroup, kBins, rows, acc,
                          [&](uint32_t r) { return tb.sums[(size_t)r * kGroups + group] != 0; });
  {
    const uint32_t c = threadIdx.x < kGroup ? acc[kGroup - 1 - threadIdx.x] : 0u;
    uint32_t total;
    const uint32_t above = over + block_exclusive_scan<uint32_t, kBlock>(c, smem, &total);
    if (above < k && k <= above + c) {
      const uint32_t bin = group * kGroup + (kGroup - 1u - threadIdx.x);
      if (sizeof(S) == 2) {
        thr[0] = bin;
        thr[1] = above + c;
      } else {
        if (FEW) {
          found[0] = bin;
          found[1] = above;
        } else {
          tb.state[0] = bin;
          tb.state[1] = k - above;
          tb.state[2] = above;
        }
      }
    }
  }
  if (sizeof(S) == 4 && !FEW && threadIdx.x < 2) tb.state[3 + threadIdx.x] = 0;
  if (FEW) {
    __shared__ uint16_t members[kFewItems * kBlock];
    __shared__ uint32_t listed;
    if (threadIdx.x == 0) listed = 0;
    __syncthreads();
    const uint32_t top = found[0], above = found[1];
#pragma unroll
    for (int i = 0; i < kItems; ++i)
      if (threadIdx.x + (uint32_t)i * kBlock < s && (key[i] >> 16) == top) members[atomicAdd(&listed, 1u)] = (uint16_t)key[i];
    __syncthreads();
    low_halves(listed, top, k - above, above, thr, [&](uint32_t j) -> uint32_t { return members[j]; });
  }
}

// fp32: the low halves of the keys in the k-th's bin (a few thousand of millions) are listed by all workgroups;
// the last one finds the k-th among them, eight bits at a time.
constexpr int kMemberItems = 8;
__global__ __launch_bounds__(kBlock) void k_sample_members(SampleTables tb, int64_t s, uint32_t *__restrict__ thr) {
  __shared__ uint16_t mine[kBlock * kMemberItems];
  __shared__ uint32_t n_mine, base;
  __shared__ bool last;
  const uint32_t top = tb.state[0];
  for (int64_t j0 = (int64_t)blockIdx.x * kBlock * kMemberItems; j0 < s; j0 += (int64_t)gridDim.x * kBlock * kMemberItems) {
    if (threadIdx.x == 0) n_mine = 0;
    __syncthreads();
    uint32_t key[kMemberItems];
#pragma unroll
    for (int i = 0; i < kMemberItems; ++i) {
      const int64_t j = j0 + threadIdx.x + (int64_t)i * kBlock;
      key[i] = j < s ? tb.sample[j] : 0xffffffffu;
    }
#pragma unroll
    for (int i = 0; i < kMemberItems; ++i)
      if ((key[i] >> 16) == top) mine[atomicAdd(&n_mine, 1u)] = (uint16_t)key[i];
    __syncthreads();
    if (threadIdx.x == 0 && n_mine) base = atomicAdd(&tb.state[3], n_mine);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n_mine; i += kBlock)
      __hip_atomic_store(&tb.members[base + i], mine[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
  }
  wait_global_acks();
  __syncthreads();
  if (threadIdx.x == 0) last = atomicAdd(&tb.state[4], 1u) == gridDim.x - 1u;
  __syncthreads();
  if (!last) return;
  const uint32_t m = load_fresh(&tb.state[3]);
  low_halves(m, top, tb.state[1], tb.state[2], thr, [&](uint32_t j) -> uint32_t {
    return __hip_atomic_load(&tb.members[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  });
}

// Workgroups of the counting kernel for a sample of s elements: one per compute unit, an element per thread at least
// (10 486 elements with four per thread 4.8 us more), more of them if a share outgrew the counters.  The picking kernel
// reads a row per workgroup, which costs less than what the counting kernel gains: counting and picking with a workgroup to
// each 4096 elements, 64 at least, and so, us: 128 660 fp32 elements on 64 and 126 workgroups 8.7 + 4.4 and 7.4 + 4.6,
// 619 534 bf16 on 152 and 256 17.8 + 6.2 and 17.2 + 6.4.
inline int64_t sample_groups(int64_t s) {
  int64_t g = ceil_div(s, (int64_t)kBlock);
  if (g > 256) g = 256;
  const int64_t least = ceil_div(s, kShare);
  return g < least ? least : g;
}

SampleTables plan_sample(void *workspace, int64_t s, int dtype, size_t *bytes) {
  Carver cv(workspace);
  SampleTables tb{};
  if (s > kOneMax) {
    const size_t g = (size_t)sample_groups(s);
    tb.state = cv.take<uint32_t>(8);
    tb.sums = cv.take<uint16_t>(g * kGroups);
    tb.bins = cv.take<uint16_t>(g * kBins);
    if (dtype == ZEN_F32) {
      tb.sample = cv.take<uint32_t>((size_t)s);
      tb.members = cv.take<uint16_t>((size_t)s);
    }
  }
  *bytes = cv.used;
  return tb;
}

template <typename S>
int sample_threshold_launch(const S *in, int64_t n, const int64_t *at, int64_t s, int64_t k, uint32_t *thr,
                            void *workspace, int32_t *status, hipStream_t stream) {
  if (s <= kOneMax) {
    k_sample_one<S><<<dim3(1), dim3(kBlock), 0, stream>>>(in, n, at, (uint32_t)s, (uint32_t)k, thr, status);
    ZEN_LAUNCH_CHECK("k_sample_one");
    return ZEN_OK;
  }
  size_t bytes;
  const SampleTables tb = plan_sample(workspace, s, sizeof(S) == 2 ? ZEN_BF16 : ZEN_F32, &bytes);
  const int64_t groups = sample_groups(s);
  const int64_t share = ceil_div(s, groups);
  const int64_t rows = ceil_div(s, share);
  k_sample_count<S><<<dim3((unsigned)rows), dim3(kBlock), 0, stream>>>(in, n, at, s, share, tb, status);
  ZEN_LAUNCH_CHECK("k_sample_count");
  const bool few = sizeof(S) == 4 && s <= kFewItems * kBlock;
  const auto pick = few ? k_sample_pick<S, sizeof(S) == 4> : k_sample_pick<S, false>;
  pick<<<dim3(1), dim3(kBlock), 0, stream>>>(tb, (uint32_t)rows, (uint32_t)s, (uint32_t)k, thr);
  ZEN_LAUNCH_CHECK("k_sample_pick");
  if (sizeof(S) == 4 && !few) {
    int64_t blocks = ceil_div(s, (int64_t)kBlock * kMemberItems);
    if (blocks > 256) blocks = 256;
    k_sample_members<<<dim3((unsigned)blocks), dim3(kBlock), 0, stream>>>(tb, s, thr);
    ZEN_LAUNCH_CHECK("k_sample_members");
  }
  return ZEN_OK;
}

}  // namespace

// The whole tensor is a sample whose positions are its own (no position array: at == nullptr).
size_t topk_whole_bytes(int64_t n, int dtype) {
  size_t bytes;
  (void)plan_sample(nullptr, n, dtype, &bytes);
  return bytes;
}

int topk_whole(const void *in, int dtype, int64_t n, int64_t k, uint32_t *thr, void *scratch, hipStream_t stream) {
  if (dtype == ZEN_BF16)
    return sample_threshold_launch(static_cast<const uint16_t *>(in), n, nullptr, n, k, thr, scratch, nullptr, stream);
  return sample_threshold_launch(static_cast<const uint32_t *>(in), n, nullptr, n, k, thr, scratch, nullptr, stream);
}

}  // namespace zen

extern "C" {

size_t zen_sample_threshold_workspace(int64_t s, int dtype) {
  if (s < 0) return 0;
  size_t bytes;
  (void)zen::plan_sample(nullptr, s, dtype, &bytes);
  return bytes > 256 ? bytes : 256;
}

int zen_sample_threshold(const void *input, int dtype, int64_t n, const int64_t *sample_index, int64_t s, int64_t k,
                         uint32_t *thr, void *workspace, size_t workspace_bytes, int32_t *status, void *stream) {
  using namespace zen;
  if (!input || !sample_index || !thr || !workspace || !status) return fail(ZEN_EINVAL, "zen_sample_threshold: null pointer");
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_sample_threshold: bad dtype");
  if (n <= 0 || s <= 0 || s > 0x7fffffffll || k < 1 || k > s)
    return fail(ZEN_EINVAL, "zen_sample_threshold: need n > 0 and 1 <= k <= s < 2^31");
  if (workspace_bytes < zen_sample_threshold_workspace(s, dtype))
    return fail(ZEN_EWORKSPACE, "zen_sample_threshold: workspace too small");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t *at = sample_index;
  if (dtype == ZEN_BF16)
    return sample_threshold_launch(static_cast<const uint16_t *>(input), n, at, s, k, thr, workspace, status, st);
  return sample_threshold_launch(static_cast<const uint32_t *>(input), n, at, s, k, thr, workspace, status, st);
}

}  // extern "C"
