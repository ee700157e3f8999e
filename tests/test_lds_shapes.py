"""LDS of the radiation-field kernel's workgroups (csrc/mgr_lds.hpp): for every
number of lines, waves per workgroup and window size the launch shape's bytes
stay within the workgroup's 64 KB, each wave's window holds what the kernel
places in it, and a window is shrunk only where the next point would not fit."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "mgr_lds.hpp"
int main()
{
    long bad = 0;
    // row and fixed bytes of the FP32 and the FP64 window
    const size_t rows[2] = {16, 32}, fixed[2] = {64 * (4 + 8 + 4), 64 * (8 + 16 + 4)};
    for (int p = 0; p < 2; p++)
        for (int L = 1; L <= 64; L++)
            for (int w = 1; w <= 4; w++)
                for (int ch = 2; ch <= 64; ch++) {
                    const size_t row = rows[p] * L, table = 8 * (size_t)L;
                    const mgr::FieldLds x = mgr::field_lds(fixed[p], row, table, w, ch);
                    const size_t need = fixed[p] + row * (x.points + 1);
                    const bool shrunk = x.points < ch;
                    const size_t next = (need + row + 63) / 64 * 64 * w + table;
                    if (x.points < 2 || x.points > ch || x.wave < need || x.wave % 64 || x.total != x.wave * w + table ||
                        x.total > 65536 || (shrunk && next <= 65536)) {
                        printf("%s L %d waves %d points %d: %d points, %zu bytes\n", p ? "fp64" : "fp32", L, w, ch,
                               x.points, x.total);
                        bad++;
                    }
                }
    return bad != 0;
}
"""


def test_every_shape_fits_the_workgroup(tmp_path):
    src, exe = tmp_path / "lds.cpp", tmp_path / "lds"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "magritte_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout[:2000]
