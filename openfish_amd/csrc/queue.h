// Where a launcher puts its kernel: a stream, and an event that the kernel's own end completes (or null).
//
// An event recorded behind a kernel is a packet of its own in the stream, and what follows waits for it as well: 3 to 4 us for each one
// between two kernels.  An event that the kernel's dispatch carries is free (three kernels of 35 us, us: 114.4 without events,
// 130.5 with two events behind each of the first two, 112.7 with one carried by each).
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

namespace {

struct Queue {
    hipStream_t stream;
    hipEvent_t done;
};

template <typename T>
struct AsDeclared {
    typedef T type;
};

// The launch's own status is left for hipGetLastError, as with a plain launch.
template <typename... P>
void queue_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, Queue queue, typename AsDeclared<P>::type... args) {
    void *argv[] = {static_cast<void *>(&args)...};
    const void *address = reinterpret_cast<const void *>(kernel);
    if (queue.done) (void)hipExtLaunchKernel(address, grid, block, argv, lds, queue.stream, nullptr, queue.done, 0);
    else (void)hipLaunchKernel(address, grid, block, argv, lds, queue.stream);
}

}  // namespace
