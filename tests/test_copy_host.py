"""Large copies to the host (csrc/mgr_copy.hip), compiled for the host with host
memory as the device's: every byte arrives at sizes around the chunk and the
threshold, whether threads start, none do (no threads left, no memory for one)
or there is no pinned memory, two copies at once both end, and an error of the
device is returned."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstddef>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0;
using hipStream_t = int;
using hipEvent_t = int *;
hipError_t hipSetDevice(int device);
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind k);
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind k, hipStream_t s);
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags);
hipError_t hipHostFree(void *p);
hipError_t hipGetLastError();
hipError_t hipStreamSynchronize(hipStream_t s);
"""

PROGRAM = r"""
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <pthread.h>
#include <dlfcn.h>
#include <thread>
#include <vector>
#include "mgr_copy.hpp"

static std::atomic<int> plain{0}, chunks{0}, fail_chunk{-1}, no_pinned{0}, threads{0}, no_threads{0};
static std::atomic<bool> no_memory{false};
static const std::thread::id first = std::this_thread::get_id();

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { plain++; std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (chunks++ == fail_chunk) return hipErrorUnknown;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new int; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (no_pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

// threads that cannot start, and memory that is not there for a thread's state
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg)
{
    if (no_threads) return EAGAIN;
    threads++;
    using create_t = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static create_t real = (create_t)dlsym(RTLD_NEXT, "pthread_create");
    return real(t, a, f, arg);
}
void *operator new(size_t n)
{
    if (no_memory && std::this_thread::get_id() == first) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static int bad = 0;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); bad = 1; } } while (0)

int main()
{
    using namespace mgr;
    const size_t S = Bounce::SLOT;
    std::vector<char> src(21 * S + 77), dst(src.size());
    for (size_t i = 0; i < src.size(); i++) src[i] = (char)(i * 2654435761u >> 13);
    auto copy = [&](Bounce &b, size_t n) {
        std::fill(dst.begin(), dst.end(), 0);
        const hipError_t e = copy_out(b, 0, 0, dst.data(), src.data(), n);
        if (e == hipSuccess) CHECK(!std::memcmp(dst.data(), src.data(), n) && (n == dst.size() || dst[n] == 0));
        return e;
    };
    {
        Bounce b;
        for (size_t n : {(size_t)0, (size_t)1, S, 2 * S - 1}) {
            plain = 0;
            CHECK(copy(b, n) == hipSuccess && plain == 1 && threads == 0);
        }
        for (size_t n : {2 * S, 2 * S + 1, 3 * S, 16 * S + 5, src.size()}) {
            plain = 0;
            CHECK(copy(b, n) == hipSuccess && plain == 0);
        }
        CHECK(threads > 0 || std::thread::hardware_concurrency() < 2);
        // no thread can start: this one does it all
        threads = 0;
        no_threads = 1;
        CHECK(copy(b, 9 * S) == hipSuccess && threads == 0);
        no_threads = 0;
        // no memory for a thread's state
        no_memory = true;
        const hipError_t e = copy_out(b, 0, 0, dst.data(), src.data(), src.size());
        no_memory = false;
        CHECK(e == hipSuccess && dst == src);
        // the device's error
        for (int k : {0, 3, 20}) {
            chunks = 0;
            fail_chunk = k;
            CHECK(copy(b, src.size()) == hipErrorUnknown);
        }
        fail_chunk = -1;
        CHECK(copy(b, src.size()) == hipSuccess);
        // two at once
        std::vector<char> other(src.size());
        std::thread t([&] { for (int i = 0; i < 20; i++) copy_out(b, 0, 0, other.data(), src.data(), src.size()); });
        for (int i = 0; i < 20; i++) CHECK(copy(b, src.size()) == hipSuccess);
        t.join();
        CHECK(other == src);
    }
    Bounce none;
    no_pinned = 1;
    plain = 0;
    CHECK(copy(none, src.size()) == hipSuccess && plain == 1);
    return bad;
}
"""


def test_on_the_host(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    csrc = os.path.join(ROOT, "magritte_amd", "csrc")
    exe = tmp_path / "copy"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", csrc, "-x", "c++",
                    os.path.join(csrc, "mgr_copy.hip"), str(tmp_path / "main.cpp"), "-o", str(exe), "-ldl"], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
