"""bench.py's roofline entry on the CPU: it says that its rate counts points that
the kernel passes over, and the hash that ties the counters to the kernel covers
every header the kernel's unit includes."""
import os
import re
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def test_the_rate_says_what_it_counts():
    import bench
    out = bench.roofline_entry(1000, 186, 100, 1.0, "fp32", "k_radiation_field<float, true>", "envelope64")
    assert "passed over" in out["note"] and "valu_issue_frac" in out["note"]
    assert out["achieved"] == round(28 * 1000 * 186 / 1e-3 / 1e12, 2)


def test_the_hash_covers_the_kernels_headers():
    import bench
    csrc = os.path.join(ROOT, "magritte_amd", "csrc")
    names = re.findall(r'#include "(mgr_[a-z]+\.hpp)"', open(os.path.join(csrc, "mgr_radiation.hip")).read())
    assert len(names) >= 3
    for name in ["mgr_radiation.hip"] + names:
        assert "magritte_amd/csrc/" + name in bench.KERNEL_SOURCES, name
