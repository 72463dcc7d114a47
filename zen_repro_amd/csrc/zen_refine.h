// The last step of an fp32 top-k threshold on the slab paths (zen_slab_encode.hip, zen_wide_encode.hip).
#pragma once

#include "zen_select.h"
#include "zen_slab_feed.h"

namespace zen {
namespace {

// --------------------------------------------- fp32: the threshold's last 16 bits

constexpr int kRefineBins = 65536;
constexpr int kRefineCoarse = kRefineBins + (int)kDoneWords;  // behind the bins: the count of finished workgroups, ...
constexpr int kRefineWords = kRefineCoarse + 256;             // ... and a counter per 256 bins
constexpr int kRefineBlock = 512;
constexpr uint32_t kRefineWaves = kRefineBlock / 64, kRefineMost = 128;  // workgroups: each ends with atomics on a few lines
// A wave to a part, or several where that leaves some without (a wave to a part alone: 5.8 us instead of 5.3 for 128 parts
// of 90 candidates; a workgroup to a part: 7.8 instead of 5.8 for 1024 of them, and two million candidates 29.6 and 23.8).
__host__ __device__ inline uint32_t refine_share(uint32_t parts) {
  const uint32_t share = kRefineMost * kRefineWaves / parts;
  return share < 1u ? 1u : share < kRefineWaves ? share : kRefineWaves;
}
inline uint32_t refine_grid(uint32_t parts) {
  const uint32_t blocks = (parts * refine_share(parts) + kRefineWaves - 1u) / kRefineWaves;
  return blocks < kRefineMost ? blocks : kRefineMost;
}

// The candidates' histogram resolves the 15 leading bits of an fp32 key: after the select kernel thr[0] is
// the lowest key of the bin the k-th largest lies in, thr[1] the number of candidates at or above it and
// *above the number in the bins above.  This kernel histograms the low 16 key bits of the candidates of that
// bin (they sit in word plane `val_plane` of the coarse slabs, or with val_plane < 0 in the second word of the
// wide buckets' two-word records; element 0, which is never handed on, is looked at in the tensor), and the
// workgroup that finishes last replaces thr[0..1] by the exact key and the number of elements at or above it.
// Grid: any number of workgroups, whose waves take the parts of the coarse slabs in turn (refine_grid).  hist: kRefineWords zeroed words.
// A chain of trips to memory bounds it.  A counter per 256 bins, gathered in LDS and handed on by every workgroup, leaves
// the last one 512 words to read: 4.8 us for 11 000 candidates, 11.8 while it read all 65 536 bins.
__global__ __launch_bounds__(kRefineBlock) void k_refine_threshold(CoarseGeom cg, int val_plane,
                                                                   const uint32_t *__restrict__ coarse_cursor,
                                                                   const uint32_t *__restrict__ coarse_words,
                                                                   const uint32_t *__restrict__ dense,
                                                                   uint32_t *thr, const uint32_t *above, uint32_t k,
                                                                   uint32_t *hist, uint32_t *thr_copy, int32_t *status) {
  __shared__ uint32_t s_scan[kRefineBlock / 64 + 1];
  __shared__ uint32_t s_coarse[256];
  __shared__ bool s_last;
  if (threadIdx.x < 256u) s_coarse[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t base = thr[0];
  const size_t plane = (size_t)cg.groups * kCoarseSplit * cg.cap;
  const uint32_t parts = cg.groups * (uint32_t)kCoarseSplit;
  const uint32_t share = refine_share(parts);  // waves to a part
  for (uint32_t unit = blockIdx.x * kRefineWaves + threadIdx.x / 64u; unit < parts * share; unit += gridDim.x * kRefineWaves) {
    const uint32_t part = unit / share;
    uint32_t count = coarse_cursor[coarse_cursor_at(part / kCoarseSplit, part % kCoarseSplit)];
    if (count > cg.cap) count = cg.cap;
    const uint32_t *vals = val_plane < 0 ? coarse_words + (size_t)part * cg.cap * 2 + 1
                                         : coarse_words + (size_t)val_plane * plane + (size_t)part * cg.cap;
    const uint32_t stride = val_plane < 0 ? 2u : 1u;
    constexpr int kAhead = 4;  // values in flight, in no branch (places past the end read the part's first)
    const uint32_t step = 64u * share;
    for (uint32_t e0 = unit % share * 64u + threadIdx.x % 64u; e0 < count; e0 += kAhead * step) {
      uint32_t v[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) v[i] = vals[(e0 + i * step < count ? e0 + i * step : e0) * stride];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const uint32_t d = (v[i] & KeyOf<uint32_t>::kMask) - base;
        if (e0 + i * step < count && d < (uint32_t)kRefineBins) {
          atomicAdd(&hist[d], 1u);
          atomicAdd(&s_coarse[d >> 8], 1u);
        }
      }
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const uint32_t key0 = dense[0] & KeyOf<uint32_t>::kMask;  // counted by the select kernel if it was a candidate
    if (key0 - base < (uint32_t)kRefineBins) {  // base is at or above the floor
      atomicAdd(&hist[key0 - base], 1u);
      atomicAdd(&s_coarse[(key0 - base) >> 8], 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x < 256u && s_coarse[threadIdx.x]) atomicAdd(&hist[kRefineCoarse + threadIdx.x], s_coarse[threadIdx.x]);
  wait_global_acks();
  __syncthreads();
  if (threadIdx.x == 0) s_last = done_last(&hist[kRefineBins], blockIdx.x, gridDim.x);
  __syncthreads();
  if (!s_last) return;
  // from the top down: the 256 bins that hold the rank, then the bin among them.  The counts were raised by atomics in
  // memory: they are read from there.
  static_assert(kRefineBlock >= 256, "a counter per thread");
  __shared__ uint32_t s_group, s_before;
  const uint32_t down = 255u - threadIdx.x;
  const uint32_t mine = threadIdx.x < 256u ? load_fresh(&hist[kRefineCoarse + down]) : 0u;
  uint32_t total;
  uint32_t before = block_exclusive_scan<uint32_t, kRefineBlock>(mine, s_scan, &total);
  const uint32_t over = above[0];
  const uint32_t need = k > over ? k - over : 1u;  // rank inside the bin of 65536 keys, from the top
  if (total < need) {
    if (threadIdx.x == 0) atomicOr(status, ZEN_STAT_RETRY);  // the two histograms disagree: let the general mode answer
    return;
  }
  if (before < need && need <= before + mine) {
    s_group = down;
    s_before = before;
  }
  __syncthreads();
  const uint32_t bin = s_group * 256u + down;
  const uint32_t here = threadIdx.x < 256u ? load_fresh(&hist[bin]) : 0u;
  const uint32_t ahead = s_before + block_exclusive_scan<uint32_t, kRefineBlock>(here, s_scan, &total);
  if (ahead < need && need <= ahead + here) {
    thr[0] = base + bin;
    thr[1] = over + ahead + here;
    if (thr_copy) {
      thr_copy[0] = base + bin;
      thr_copy[1] = over + ahead + here;
    }
  }
}

}  // namespace
}  // namespace zen
