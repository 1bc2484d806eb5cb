// status.hip — the host's one look at a launch: whether any row's status bit is set, and whether
// any id lies outside its range.
//
// The sampler and scoring calls raise the reference's ValueErrors (dsv41_train/rl/rollout.py:145-146,
// models/dsv4/model.py:725-727), so every checked call ends with this question.  Asked with
// tensor operations it took a compare, a reduction and a copy back behind the launch, and the
// host's wake-up from its wait: 15 us of the 75 us of an 8-row call.  Here one workgroup answers
// into pinned memory that the host watches.  (An empty launch and hipStreamSynchronize take
// 11.4 us on this machine, a launch and a watched word 6.0.)  Bound by its loads' latency up to a
// few thousand values, then by what one CU reads: 1000000 statuses 38 us a call with four 16-byte
// loads in flight per thread (114 with single ones), 30 by tensor operations, which the Python
// calls use above 2^18.

#include <chrono>

#include "common.h"

namespace dsv41 {
namespace status {

constexpr int NT = 1024;
// how long the host watches before it waits on the stream (and learns of a failed launch)
constexpr std::chrono::microseconds WATCH{2000};

// Whether pred holds for some a[i] of the n values: 16-byte loads, four in flight per thread, with
// single ones before the first 16-byte boundary and behind the last.
template <typename T, class Pred>
__device__ __forceinline__ bool any_of(const T* a, int64_t n, Pred pred) {
  constexpr int G = 16 / (int)sizeof(T), U = 4;
  struct alignas(16) Group {
    T v[G];
  };
  if (n <= NT) return threadIdx.x < n && pred(a[threadIdx.x]);  // 2.4 us, 2.7 the general way
  bool hit = false;
  const int64_t head = min(n, (int64_t)((16 - ((uintptr_t)a & 15)) & 15) / (int)sizeof(T));
  if (threadIdx.x < head) hit |= pred(a[threadIdx.x]);
  const Group* g = reinterpret_cast<const Group*>(a + head);
  const int64_t groups = (n - head) / G;
  int64_t i = threadIdx.x;
  for (; i + (U - 1) * NT < groups; i += U * NT) {
    Group x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = g[i + u * NT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < G; ++k) hit |= pred(x[u].v[k]);
  }
  for (; i < groups; i += NT) {
    const Group x = g[i];
#pragma unroll
    for (int k = 0; k < G; ++k) hit |= pred(x.v[k]);
  }
  const int64_t tail = head + groups * G + threadIdx.x;
  if (tail < n) hit |= pred(a[tail]);
  return hit;
}

// flags[0]: 1 + (1 if some status is set) + (2 if some id lies outside [0, limit)).
__global__ __launch_bounds__(NT) void check_kernel(const int32_t* st, int64_t n, const int64_t* ids, int64_t n_ids,
                                                   int64_t limit, int32_t* flags) {
  const int set = __syncthreads_or(any_of(st, n, [](int32_t s) { return s != 0; }));
  const int outside =
      __syncthreads_or(any_of(ids, n_ids, [=](int64_t t) { return (uint64_t)t >= (uint64_t)max(limit, (int64_t)0); }));
  if (threadIdx.x == 0)
    __hip_atomic_store(flags, 1 + (set ? 1 : 0) + (outside ? 2 : 0), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace status
}  // namespace dsv41

using namespace dsv41;

extern "C" int dsv41_check_wait(const int32_t* st, int64_t n, const int64_t* ids, int64_t n_ids, int64_t limit,
                                int32_t* flags, void* stream) {
  if (n < 0 || n_ids < 0 || (n > 0 && !st) || (n_ids > 0 && !ids) || !flags)
    return fail(DSV41_E_INVALID, "check: statuses, ids and flags are required");
  hipStream_t s = static_cast<hipStream_t>(stream);
  __atomic_store_n(flags, 0, __ATOMIC_RELAXED);
  hipLaunchKernelGGL(status::check_kernel, dim3(1), dim3(status::NT), 0, s, st, n, ids, n_ids, limit, flags);
  DSV41_HIP_CHECK(hipGetLastError());
  const auto until = std::chrono::steady_clock::now() + status::WATCH;
  int got = 0;
  do {
    for (int i = 0; i < 64 && got == 0; ++i) got = __atomic_load_n(flags, __ATOMIC_ACQUIRE);
  } while (got == 0 && std::chrono::steady_clock::now() < until);
  if (got == 0) {
    DSV41_HIP_CHECK(hipStreamSynchronize(s));
    got = __atomic_load_n(flags, __ATOMIC_ACQUIRE);
    if (got == 0) return fail(DSV41_E_HIP, "check: the launch left no answer");
  }
  return got - 1;
}
