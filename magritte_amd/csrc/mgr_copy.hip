// mgr_copy.hip -- large copies to the host through pinned staging memory (host
// code only).
#include "mgr_copy.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

using namespace mgr;

bool Bounce::allocate()
{
    if (slots) return true;
    for (auto &e : event)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
    return hipHostMalloc((void **)&slots, WORKERS * SLOT, hipHostMallocDefault) == hipSuccess;
}

Bounce::~Bounce()
{
    for (auto e : event)
        if (e) (void)hipEventDestroy(e);
    if (slots) (void)hipHostFree(slots);
}

// Chunks of a copy to the host, each claimed by one worker: to its pinned slot
// by the copy engine, and on to dst while other workers' chunks are on their way.
static hipError_t copy_chunks(Bounce &b, int device, hipStream_t stream, int worker, std::atomic<size_t> &next,
                              char *dst, const char *src, size_t bytes)
{
    hipError_t e = hipSetDevice(device);
    char *slot = b.slots + worker * b.SLOT;
    for (size_t off; e == hipSuccess && (off = next.fetch_add(b.SLOT)) < bytes;) {
        const size_t n = std::min(b.SLOT, bytes - off);
        e = hipMemcpyAsync(slot, src + off, n, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(b.event[worker], stream);
        if (e == hipSuccess) e = hipEventSynchronize(b.event[worker]);
        if (e == hipSuccess) std::memcpy(dst + off, slot, n);
    }
    return e;
}

// Into pageable memory a plain copy is bound by one thread that moves the data
// and takes the page faults of a fresh array: 139 MB at 17 GB/s (4.5 fresh);
// with up to 8 threads 38 GB/s (22 fresh).  Below 4 MB starting the threads
// costs what they gain (4 MB: 0.24 ms plain, 0.19 so; 1 MB: 0.07 and 0.09).
hipError_t mgr::copy_out(Bounce &b, int device, hipStream_t stream, void *dst, const void *src, size_t bytes)
{
    if (bytes >= 2 * Bounce::SLOT) {
        std::unique_lock<std::mutex> mine(b.busy, std::try_to_lock);   // another thread's copy goes on by itself
        if (mine && b.allocate()) {
            std::atomic<size_t> next{0};
            std::atomic<int> failed{0};
            auto work = [&](int worker) {
                const hipError_t e = copy_chunks(b, device, stream, worker, next, static_cast<char *>(dst),
                                                 static_cast<const char *>(src), bytes);
                if (e != hipSuccess) failed = (int)e;
            };
            const int workers = (int)std::min<size_t>({(size_t)Bounce::WORKERS, (bytes + Bounce::SLOT - 1) / Bounce::SLOT,
                                                       std::max<size_t>(1, std::thread::hardware_concurrency())});
            std::thread th[Bounce::WORKERS];
            try {
                for (int w = 1; w < workers; w++) th[w] = std::thread(work, w);
            } catch (const std::exception &) {   // no more threads, or no memory for one: those there are do it all
            }
            work(0);
            for (auto &t : th)
                if (t.joinable()) t.join();
            if (failed) (void)hipStreamSynchronize(stream);   // no copy into the slots goes on
            return (hipError_t)failed.load();
        }
        if (mine) (void)hipGetLastError();   // no staging memory: the plain copy
    }
    return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
}
