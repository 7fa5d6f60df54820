// Whether the kernels of two streams run side by side.
//
// The runtime deals the streams of a process round its few hardware queues (four unless the environment says
// otherwise, the null stream's among them), and kernels of one queue run one after another whatever streams they
// are on.  Nothing in the API tells which queue a stream got, so it is tried: one lane on the first stream waits
// for the mark that one lane on the second sets.  In one queue the mark comes after the wait has ended.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace {

// 100 us of the 100 MHz clock; the other kernel is launched right behind this one and starts within 10 to 20.
// The number of polls bounds the wait by itself (a poll of host memory takes a microsecond or two).
constexpr long long kWaitTicks = 10000;
constexpr int kWaitPolls = 2000;

// mark: two ints of pinned host memory, both zero before the launches; mark[0] arrived, mark[1] seen in time
__global__ void meet_kernel(int *mark, int waits) {
    if (!waits) {
        __hip_atomic_store(mark, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    const long long start = wall_clock64();
    int seen = 0;
    for (int k = 0; k < kWaitPolls && !seen && wall_clock64() - start < kWaitTicks; ++k)
        seen = __hip_atomic_load(mark, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(mark + 1, seen, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

extern "C" int ofk_meet(int *mark, int waits, void *stream) {
    if (!mark) return OFK_BAD_ARGS;
    hipLaunchKernelGGL(meet_kernel, dim3(1), dim3(1), 0, static_cast<hipStream_t>(stream), mark, waits);
    return (int)hipGetLastError();
}
