"""Device memory kept between models (csrc/mgr_blocks.hip), compiled for the host
with a device of 8 GB whose allocations are counted: an allocation of any kind
that does not fit takes the kept blocks back, at most 2 GB are kept, the oldest
go first, a block goes to an allocation of 4/5 of its size or more on its own
device, and nothing is leaked, also from several threads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstddef>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
using hipStream_t = int;   // 0: idle
hipError_t hipMalloc(void **p, size_t bytes);
hipError_t hipFree(void *p);
hipError_t hipGetLastError();
hipError_t hipStreamSynchronize(hipStream_t s);
"""

PROGRAM = r"""
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>
#include <vector>
#include "mgr_blocks.hpp"

static std::mutex lock;
static std::map<void *, size_t> live;
static size_t in_use = 0, next_p = 4096;
static thread_local hipError_t last = hipSuccess;
static const size_t GB = (size_t)1 << 30, CARD = 8 * GB;

hipError_t hipMalloc(void **p, size_t bytes)
{
    std::lock_guard<std::mutex> l(lock);
    if (bytes > CARD - in_use) return last = hipErrorOutOfMemory;
    *p = (void *)next_p;
    next_p += bytes + 4096;
    live[*p] = bytes;
    in_use += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> l(lock);
    if (!live.count(p)) return last = hipErrorUnknown;
    in_use -= live[p];
    live.erase(p);
    return hipSuccess;
}
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipStreamSynchronize(hipStream_t s) { return s ? hipErrorUnknown : hipSuccess; }

static int bad = 0;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); bad = 1; } } while (0)

int main()
{
    using namespace mgr;
    void *a, *b, *c, *d;
    // a plain allocation takes the kept memory back
    CHECK(block_malloc(0, &a, GB) == hipSuccess && block_malloc(0, &b, GB / 2) == hipSuccess);
    block_free(0, a);
    block_free(0, b);
    CHECK(blocks_kept(0) == GB + GB / 2 && in_use == blocks_kept(0) && blocks_kept(1) == 0);
    CHECK(device_malloc(&c, 6 * GB) == hipSuccess && blocks_kept(0) == GB + GB / 2);
    CHECK(device_malloc(&d, 2 * GB) == hipSuccess && blocks_kept(0) == 0 && in_use == CARD);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(device_malloc(&a, 1) == hipErrorOutOfMemory && a == nullptr && hipGetLastError() == hipSuccess);
    CHECK(block_malloc(0, &a, GB) == hipErrorOutOfMemory && hipGetLastError() == hipSuccess);
    hipFree(c);
    hipFree(d);
    // reuse: the smallest kept block of 1 to 5/4 of the size, on its device
    const size_t H = GB / 2;
    CHECK(block_malloc(0, &a, H) == hipSuccess && block_malloc(0, &b, H + H / 8) == hipSuccess);
    block_free(0, b);
    block_free(0, a);
    CHECK(block_malloc(1, &c, H) == hipSuccess && c != a && c != b);
    CHECK(block_malloc(0, &d, H / 2) == hipSuccess && d != a && d != b);
    hipFree(d);
    CHECK(block_malloc(0, &d, H) == hipSuccess && d == a);
    CHECK(block_malloc(0, &a, H) == hipSuccess && a == b);
    CHECK(blocks_kept(0) == 0);
    block_free(0, a);
    block_free(0, c);
    CHECK(blocks_kept(0) == H + H / 8 && blocks_kept(1) == H);
    block_free(1, d);   // a stream in error: not kept
    CHECK(blocks_kept(0) == H + H / 8);
    // above 2 GB the oldest goes
    CHECK(block_malloc(0, &d, GB) == hipSuccess);
    block_free(0, d);
    CHECK(blocks_kept(0) == GB && blocks_kept(1) == H);
    CHECK(block_malloc(0, &d, GB) == hipSuccess);
    block_free(0, d);
    // on request
    CHECK(blocks_release() == GB + H && blocks_release() == 0 && in_use == 0);
    // larger than all that is kept, and small ones: plain
    CHECK(block_malloc(0, &a, 3 * GB) == hipSuccess && block_malloc(0, &b, 1 << 20) == hipSuccess);
    block_free(0, a);
    block_free(0, b);
    CHECK(in_use == 0 && blocks_release() == 0);
    // threads that fill the card by turns
    std::vector<std::thread> th;
    for (int t = 0; t < 8; t++)
        th.emplace_back([t] {
            for (int i = 0; i < 2000; i++) {
                void *p = nullptr, *q = nullptr;
                const size_t n = (size_t)(1 + (i * 7 + t * 3) % 9) * (GB / 8);
                if (block_malloc(0, &p, n) == hipSuccess) block_free(0, p);
                if (device_malloc(&q, n) == hipSuccess) hipFree(q);
                if (i % 97 == 0) blocks_release();
            }
        });
    for (auto &t : th) t.join();
    CHECK(blocks_kept(0) == in_use && in_use <= 2 * GB);
    blocks_release();
    CHECK(in_use == 0 && live.empty());
    return bad;
}
"""


def test_on_the_host(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    csrc = os.path.join(ROOT, "magritte_amd", "csrc")
    exe = tmp_path / "blocks"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", csrc, "-x", "c++",
                    os.path.join(csrc, "mgr_blocks.hip"), str(tmp_path / "main.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr


def test_every_allocation_goes_through():
    """No other unit calls hipMalloc itself."""
    csrc = os.path.join(ROOT, "magritte_amd", "csrc")
    for name in sorted(os.listdir(csrc)):
        if name.endswith((".hip", ".hpp")) and not name.startswith("mgr_blocks"):
            assert "hipMalloc(" not in open(os.path.join(csrc, name)).read(), name
