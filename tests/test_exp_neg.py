"""exp_neg and profile64 of the radiation-field unit, compiled for the host:
exp(-t) to 2^-52 over the range the profiles need, exactly 0 beyond it, NaN for
NaN, and no conversion of a value an int cannot hold (the compiler's check for
that is on; nearest_int, one instruction on the GPU, is written out), at any
distance from a line."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cmath>
#include <cstdio>
#include <climits>
#include <limits>
#define __device__
#define __forceinline__ inline
template <typename real> struct Prec;
template <> struct Prec<double> { static double rcp(double x) { return 1.0 / x; } };
static int nearest_int(double x)
{
    if (x != x) return 0;
    return x <= INT_MIN ? INT_MIN : x >= INT_MAX ? INT_MAX : (int)x;
}
constexpr double INVERSE_SQRT_PI = 0.5 * 1.12837916709551257390;
%s
int main()
{
    int bad = 0;
    double worst = 0.0;
    for (double t = 0.0; t < 707.0; t += 1.0 / 1024 + t * 1e-4) {
        const long double e = expl(-(long double)t);
        worst = fmax(worst, (double)fabsl((exp_neg(t) - e) / e));
        if (exp_neg(t, true) != exp_neg(t)) { printf("in at %%g\n", t); bad = 1; break; }
    }
    if (!(worst <= 0x1p-52)) { printf("relative error %%g\n", worst); bad = 1; }
    for (double t = 746.0; t < 1.0e40; t *= 1.01)
        if (exp_neg(t) != 0.0) { printf("exp_neg(%%g) = %%g\n", t, exp_neg(t)); bad = 1; break; }
    for (double t = 1.0; t < 1.0e40; t *= 1.3)
        if (exp_neg(t, false) != 0.0) { printf("out at %%g: %%g\n", t, exp_neg(t, false)); bad = 1; break; }
    if (!std::isnan(exp_neg(std::numeric_limits<double>::quiet_NaN())) ||
        !std::isnan(exp_neg(std::numeric_limits<double>::quiet_NaN(), false))) { printf("NaN\n"); bad = 1; }
    // a line's profile from its centre to 1e7 widths away
    const double width = 1.0e5;
    for (double x = 0.0; x < 1.0e7; x = x * 1.01 + 1e-3) {
        const double e = exp(-x * x) * INVERSE_SQRT_PI / width, p = profile64(width, x * width);
        if (!(fabs(p - e) <= 1e-13 * (1 + x * x) * e + 1e-320)) { printf("profile at %%g: %%g\n", x, p); bad = 1; break; }
    }
    if (!std::isnan(profile64(width, std::numeric_limits<double>::quiet_NaN()))) { printf("NaN profile\n"); bad = 1; }
    return bad;
}
"""


def test_on_the_host(tmp_path):
    text = open(os.path.join(ROOT, "magritte_amd", "csrc", "mgr_radiation.hip")).read()
    parts = re.findall(r"__device__ __forceinline__ double (?:exp_neg_parts|exp_neg|profile64)\(.*?\n}\n", text, re.S)
    assert len(parts) == 4
    src, exe = tmp_path / "exp_neg.cpp", tmp_path / "exp_neg"
    src.write_text(PROGRAM % "\n".join(parts))
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-Wno-unknown-pragmas",
                    "-fsanitize=float-cast-overflow", "-fno-sanitize-recover=all", str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
