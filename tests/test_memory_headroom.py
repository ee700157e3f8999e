"""What only saves time (the spans of sub-points, the far-end cache) leaves a quarter
of the device memory free (csrc/mgr_blocks.hpp), compiled for the host: each by
itself, and both together, whichever share of the memory the first one took."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = """
#pragma once
#include <cstddef>
enum hipError_t { hipSuccess = 0 };
using hipStream_t = int;
"""

PROGRAM = r"""
#include "mgr_blocks.hpp"
using mgr::leaves_quarter;
constexpr size_t M = (size_t)1 << 20, G = 1024 * M;
static_assert(leaves_quarter(0, 0, 0) && !leaves_quarter(1, 0, 0), "no memory");
static_assert(leaves_quarter(3 * G, 0, 4 * G) && !leaves_quarter(3 * G + 1, 0, 4 * G), "one of them");
int main()
{
    // the first takes its share of 288 GB, the second what is allowed beside it
    const size_t all = 288 * G;
    for (size_t first = 0; first <= all; first += 64 * M) {
        if (leaves_quarter(first, 0, all) != (first <= 216 * G)) return 1;
        if (first > 216 * G) continue;
        const size_t most = 216 * G - first;
        if (!leaves_quarter(most, first, all - first) || leaves_quarter(most + 1, first, all - first)) return 2;
    }
    return 0;
}
"""


def test_a_quarter_stays_free(tmp_path):
    hip = tmp_path / "hip"
    hip.mkdir()
    (hip / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "headroom")
    subprocess.run(["g++", "-std=c++17", "-I", str(tmp_path), "-I", os.path.join(ROOT, "magritte_amd", "csrc"),
                    str(tmp_path / "main.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe], timeout=60).returncode == 0


def test_both_allocations_ask():
    """The rule is what the spans and the cache are allocated by."""
    for name, call in (("mgr_trace.hip", "leaves_quarter(bytes, 0,"), ("mgr_radiation.hip", "leaves_quarter(bytes, spans,")):
        with open(os.path.join(ROOT, "magritte_amd", "csrc", name)) as f:
            assert f.read().count(call) == 1, name
