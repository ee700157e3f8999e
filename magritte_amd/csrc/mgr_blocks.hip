// mgr_blocks.hip -- device memory: large blocks kept for the next model, and
// allocations that take them back (host code only).
#include "mgr_blocks.hpp"

#include <mutex>
#include <new>
#include <vector>

// Device memory of the trace and its caches, kept for the next trace or context
// of the process when it is given back: a model's arrays are a few large blocks,
// allocated and freed once per model, and the runtime clears and unmaps every
// one: a 27^3-cell solve frees 1.6 GB and takes 30 ms, 66 to 96 while the
// clearing of larger models freed before holds the frees up; with the blocks
// kept 27 in both cases.  At most KEPT bytes are kept, the oldest go first; all
// go when an allocation of the library fails (device_malloc) or on request
// (blocks_release).  The next owner of a block writes all that it reads.
namespace {
struct Blocks {
    static constexpr size_t LEAST = 4 << 20;     // smaller ones are not kept
    static constexpr size_t KEPT = (size_t)2 << 30;
    struct Block {
        void  *p;
        size_t bytes;
        int    device;
    };
    std::mutex         m;
    std::vector<Block> kept;   // oldest first
    std::vector<Block> used;
    size_t             held = 0;

    static Blocks &get()
    {
        static Blocks *b = new Blocks;   // never destroyed: the runtime may be gone by then
        return *b;
    }

    // with m held
    size_t release()
    {
        const size_t bytes = held;
        for (const auto &k : kept) (void)hipFree(k.p);
        kept.clear();
        held = 0;
        return bytes;
    }
    // the error is the caller's: none is left for the next launch's check
    static hipError_t plain(void **p, size_t bytes)
    {
        const hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            *p = nullptr;
        }
        return e;
    }
    hipError_t allocate(void **p, size_t bytes)
    {
        hipError_t e = plain(p, bytes);
        if (e != hipSuccess && !kept.empty()) {
            release();
            e = plain(p, bytes);
        }
        return e;
    }
};
}  // namespace

hipError_t mgr::device_malloc(void **p, size_t bytes)
{
    if (Blocks::plain(p, bytes) == hipSuccess) return hipSuccess;   // without the lock as long as there is memory
    Blocks &b = Blocks::get();
    std::lock_guard<std::mutex> lock(b.m);
    return b.allocate(p, bytes);
}

hipError_t mgr::block_malloc(int device, void **p, size_t bytes)
{
    if (bytes < Blocks::LEAST) return device_malloc(p, bytes);
    Blocks &b = Blocks::get();
    try {
        std::lock_guard<std::mutex> lock(b.m);
        b.used.reserve(b.used.size() + 1);
        size_t best = b.kept.size();
        for (size_t i = 0; i < b.kept.size(); i++)
            if (b.kept[i].device == device && b.kept[i].bytes >= bytes && b.kept[i].bytes <= bytes + bytes / 4 &&
                (best == b.kept.size() || b.kept[i].bytes < b.kept[best].bytes))
                best = i;
        if (best < b.kept.size()) {
            *p = b.kept[best].p;
            b.used.push_back(b.kept[best]);
            b.held -= b.kept[best].bytes;
            b.kept.erase(b.kept.begin() + best);
            return hipSuccess;
        }
        const hipError_t e = b.allocate(p, bytes);
        if (e == hipSuccess) b.used.push_back({*p, bytes, device});
        return e;
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    }
}

size_t mgr::blocks_kept(int device)
{
    Blocks &b = Blocks::get();
    std::lock_guard<std::mutex> lock(b.m);
    size_t bytes = 0;
    for (const auto &k : b.kept)
        if (k.device == device) bytes += k.bytes;
    return bytes;
}

size_t mgr::blocks_release()
{
    Blocks &b = Blocks::get();
    std::lock_guard<std::mutex> lock(b.m);
    return b.release();
}

void mgr::block_free(hipStream_t stream, void *p)
{
    if (!p) return;
    Blocks &b = Blocks::get();
    const bool idle = hipStreamSynchronize(stream) == hipSuccess;
    try {
        std::lock_guard<std::mutex> lock(b.m);
        for (size_t i = 0; i < b.used.size(); i++) {
            if (b.used[i].p != p) continue;
            const Blocks::Block mine = b.used[i];
            if (idle && mine.bytes <= Blocks::KEPT) {
                while (b.held + mine.bytes > Blocks::KEPT) {
                    (void)hipFree(b.kept.front().p);
                    b.held -= b.kept.front().bytes;
                    b.kept.erase(b.kept.begin());
                }
                b.kept.push_back(mine);
                b.held += mine.bytes;
                p = nullptr;
            }
            b.used.erase(b.used.begin() + i);
            break;
        }
    } catch (const std::bad_alloc &) {
    }
    if (p) (void)hipFree(p);
}
