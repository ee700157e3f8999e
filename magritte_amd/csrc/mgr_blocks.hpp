// mgr_blocks.hpp -- device memory: large blocks kept for the next model, and
// allocations that take them back.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace mgr {

// hipMalloc on the current device; when it fails all kept blocks are given back
// and it is tried again.  Every device allocation of the library goes through here.
hipError_t device_malloc(void **p, size_t bytes);
template <typename T>
hipError_t device_malloc(T **p, size_t bytes)
{
    return device_malloc((void **)p, bytes);
}

// A block of the trace's arrays and caches on the current device, `device`: a kept
// one of up to 5/4 of the size, or a new one.
hipError_t block_malloc(int device, void **p, size_t bytes);
// Given back when the stream, on which alone it was used, is idle.
void       block_free(hipStream_t stream, void *p);

// What only saves time is allocated where a quarter of the memory stays free for what
// is needed: `bytes` more beside `taken` of it already there, `available` bytes being
// free or kept.
constexpr bool leaves_quarter(size_t bytes, size_t taken, size_t available)
{
    return bytes + taken <= (available + taken) / 4 * 3;
}

size_t blocks_kept(int device);   // bytes that device_malloc gives back before it fails
size_t blocks_release();          // gives all of them back now; how many bytes they had

}  // namespace mgr
