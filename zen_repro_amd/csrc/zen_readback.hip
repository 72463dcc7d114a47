// What a call has to know on the host before it can go on (split sizes, counts, status words), and the count of
// the entries a selection will have.
//
// A torch tensor's .tolist() costs a conversion, a concatenation, a copy kernel and the runtime's own wait, some
// 40 us of a small call.  Here one workgroup gathers the words from where the kernels before it left them and
// stores them, widened to 64 bits, into pinned host memory; the host watches the word that is stored last.  Where one
// of a call's own kernels knows the answer, that kernel stores it (HostAnswer, zen_common.h), and this one is not
// launched.  Each
// of the two waits of a 1 Mi-element bucket's all-reduce got 13 us shorter by it (218 -> 191 us), and with the
// counting kernel below in place of a library reduction the load balance of a 12.9 M-element fp32 tensor of
// unknown density went from 242 to 178 us, before the counting kernel had 256 workgroups.
#include <immintrin.h>  // host pass: _mm_pause

#include <chrono>
#include <thread>

#include "zen_select.h"

namespace zen {
namespace {

struct ReadBack {
  const void *from[ZEN_READ_BACK_SEGMENTS];
  int32_t count[ZEN_READ_BACK_SEGMENTS];
  int32_t wide[ZEN_READ_BACK_SEGMENTS];  // 64-bit words (else 32)
};

constexpr std::chrono::nanoseconds kSpin(1000000), kNap(1000000);

__global__ void k_read_back(ReadBack r, int64_t *host, int64_t ticket) {
  int at = 1;
#pragma unroll
  for (int s = 0; s < ZEN_READ_BACK_SEGMENTS; ++s) {
    for (int i = threadIdx.x; i < r.count[s]; i += blockDim.x)
      host_store(host + at + i, r.wide[s] ? static_cast<const int64_t *>(r.from[s])[i]
                                          : (int64_t) static_cast<const int32_t *>(r.from[s])[i]);
    at += r.count[s];
  }
  host_answered(HostAnswer{host, ticket});
}

// Elements with key >= max(thr[0], 1) (thr == nullptr: the nonzero ones).  Bound by the one read of the tensor:
// four vectors per thread are in flight, a workgroup adds up in registers and touches the counter once.  One address
// takes an add every ten nanoseconds, so there are few workgroups: 12.9 M fp32 elements 10.3 us, 62 M bf16 20.8 (1024
// workgroups of 512 threads, whose adds queue up: 19.3 and 24.5).
constexpr int kCountBlock = 1024, kCountVecs = 4;

template <typename S, bool ALIGNED>
__global__ __launch_bounds__(kCountBlock) void k_count(const S *__restrict__ in, int64_t n,
                                                       const uint32_t *__restrict__ thr,
                                                       unsigned long long *__restrict__ count) {
  constexpr int V = VecOf<S>::kN;
  __shared__ uint32_t part[kCountBlock / 64];
  uint32_t least = thr ? thr[0] : 0u;
  if (least == 0) least = 1;
  const int64_t nvec = (n + V - 1) / V;
  uint32_t mine = 0;
  for (int64_t v0 = (int64_t)blockIdx.x * kCountBlock * kCountVecs + threadIdx.x; v0 < nvec;
       v0 += (int64_t)gridDim.x * kCountBlock * kCountVecs) {
    S e[kCountVecs][V];
#pragma unroll
    for (int j = 0; j < kCountVecs; ++j) load_vec<S, ALIGNED>(in, (v0 + (int64_t)j * kCountBlock) * V, n, e[j]);
#pragma unroll
    for (int j = 0; j < kCountVecs; ++j)
#pragma unroll
      for (int i = 0; i < V; ++i) mine += uint32_t(e[j][i] & KeyOf<S>::kMask) >= least;
  }
  mine = wave_sum(mine);
  if (lane_id() == 0) part[threadIdx.x >> 6] = mine;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t sum = 0;
#pragma unroll
    for (int w = 0; w < kCountBlock / 64; ++w) sum += part[w];
    if (sum) atomicAdd(count, (unsigned long long)sum);
  }
}

template <typename S>
void launch_count(const S *in, int64_t n, const uint32_t *thr, int64_t *count, hipStream_t s) {
  const int64_t per = (int64_t)kCountBlock * kCountVecs * VecOf<S>::kN;
  int64_t blocks = ceil_div(n, per);
  if (blocks > 256) blocks = 256;  // one per compute unit
  unsigned long long *c = reinterpret_cast<unsigned long long *>(count);
  if ((reinterpret_cast<uintptr_t>(in) & 15u) == 0)
    k_count<S, true><<<dim3((unsigned)blocks), dim3(kCountBlock), 0, s>>>(in, n, thr, c);
  else
    k_count<S, false><<<dim3((unsigned)blocks), dim3(kCountBlock), 0, s>>>(in, n, thr, c);
}

}  // namespace

int host_ask(int64_t *host, int64_t words, int64_t need, HostAnswer *answer) {
  if (!host || words < need + 1) return fail(ZEN_EINVAL, "host words missing or too few");
  answer->host = host;
  answer->ticket = host[0] + 1;
  return ZEN_OK;
}

static int read_back_launch(const ReadBack &r, const HostAnswer &answer, hipStream_t s) {
  k_read_back<<<dim3(1), dim3(64), 0, s>>>(r, answer.host, answer.ticket);
  ZEN_LAUNCH_CHECK("k_read_back");
  return ZEN_OK;
}

int host_answer_launch(const HostAnswer &answer, const int64_t *first, int n0, const int32_t *second, int n1, hipStream_t s) {
  return read_back_launch(ReadBack{{first, second, nullptr}, {n0, n1, 0}, {1, 0, 0}}, answer, s);
}

static int host_wait(const HostAnswer &answer, hipStream_t s) {
  // The waits of a call are short: this core watches for the answer.  A longer one is for what the stream has to wait
  // for itself (an exchange, other ranks): then the core is left to others, for a sixteenth of the time waited so far
  // and a millisecond at most, and the stream is asked every time, which says when something on it has failed.  (The
  // runtime's own waits keep the core busy from beginning to end, hipEventBlockingSync or not.)
  using clock = std::chrono::steady_clock;
  const auto begin = clock::now();
  for (uint32_t spins = 1;; ++spins) {
    if (__atomic_load_n(answer.host, __ATOMIC_ACQUIRE) == answer.ticket) return ZEN_OK;
    _mm_pause();
    if ((spins & 63u) == 0 && clock::now() - begin > kSpin) break;
  }
  for (;;) {
    const auto nap = (clock::now() - begin) / 16;
    std::this_thread::sleep_for(nap < kNap ? nap : kNap);
    if (__atomic_load_n(answer.host, __ATOMIC_ACQUIRE) == answer.ticket) return ZEN_OK;
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady) continue;
    ZEN_HIP_CHECK(e);
    return __atomic_load_n(answer.host, __ATOMIC_ACQUIRE) == answer.ticket
               ? ZEN_OK
               : fail(ZEN_EHIP, "zen_read_back: the stream ended without an answer");
  }
}

int host_finish(int rc, const HostAnswer &answer, hipStream_t s) {
  if (rc == ZEN_OK) return host_wait(answer, s);
  // The kernel with the answer may have been launched all the same (one behind it failed, or the error was an older
  // one): its ticket is the next call's too, so it has to be there before this one returns.
  if (rc == ZEN_EHIP) (void)hipStreamSynchronize(s);
  return rc;
}

}  // namespace zen

extern "C" {

int zen_host_words_alloc(int64_t words, int64_t **host) {
  using namespace zen;
  if (!host || words < 1 || words > (1 << 20)) return fail(ZEN_EINVAL, "zen_host_words_alloc: bad size");
  void *p = nullptr;
  ZEN_HIP_CHECK(hipHostMalloc(&p, (size_t)words * sizeof(int64_t), hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent));
  *host = static_cast<int64_t *>(p);
  (*host)[0] = 0;
  return ZEN_OK;
}

int zen_host_words_free(int64_t *host) {
  using namespace zen;
  if (host) ZEN_HIP_CHECK(hipHostFree(host));
  return ZEN_OK;
}

int zen_read_back(const void *p0, int n0, int wide0, const void *p1, int n1, int wide1, const void *p2, int n2,
                  int wide2, int64_t *host, int64_t words, void *stream) {
  using namespace zen;
  ReadBack r{{p0, p1, p2}, {n0, n1, n2}, {wide0, wide1, wide2}};
  int64_t total = 1;
  for (int i = 0; i < ZEN_READ_BACK_SEGMENTS; ++i) {
    if (r.count[i] < 0 || (r.count[i] > 0 && !r.from[i])) return fail(ZEN_EINVAL, "zen_read_back: bad segment");
    total += r.count[i];
  }
  if (!host || total > words) return fail(ZEN_EINVAL, "zen_read_back: host buffer missing or too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const HostAnswer answer{host, host[0] + 1};
  return host_finish(read_back_launch(r, answer, s), answer, s);
}

int zen_count(const void *input, int dtype, int64_t n, const uint32_t *thr, int64_t *count, void *stream) {
  using namespace zen;
  if (dtype != ZEN_F32 && dtype != ZEN_BF16) return fail(ZEN_EINVAL, "zen_count: bad dtype");
  if (n < 0 || n > 0x7fffffffll || !count || (n > 0 && !input)) return fail(ZEN_EINVAL, "zen_count: bad argument");
  if (n == 0) return ZEN_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == ZEN_BF16)
    launch_count(static_cast<const uint16_t *>(input), n, thr, count, s);
  else
    launch_count(static_cast<const uint32_t *>(input), n, thr, count, s);
  ZEN_LAUNCH_CHECK("k_count");
  return ZEN_OK;
}

}  // extern "C"
