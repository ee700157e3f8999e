// mgr_copy.hpp -- large copies to the host through pinned staging memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace mgr {

// Pinned staging memory of a context for large copies to the host, allocated by
// the first one: a slot and an event for each worker.
struct Bounce {
    static constexpr size_t SLOT = 2 << 20;
    static constexpr int    WORKERS = 8;
    std::mutex busy;   // held by the copy that uses the slots
    char      *slots = nullptr;
    hipEvent_t event[WORKERS] = {};

    bool allocate();
    ~Bounce();
};

// Device to host memory, complete on return; the stream, the context's, is idle.
// No exception leaves it.
hipError_t copy_out(Bounce &b, int device, hipStream_t stream, void *dst, const void *src, size_t bytes);

}  // namespace mgr
