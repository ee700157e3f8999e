"""Device memory kept by closed contexts: given back on request, and by itself when
an allocation of the library does not fit, whatever it is for."""
import ctypes as C

import numpy as np
import pytest

from magritte_amd import hip
from magritte_amd.setup import synthetic

pytestmark = pytest.mark.gpu


def _free():
    rt = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _solve():
    ctx = hip.Context(synthetic.envelope_model(n=20, seed=1)).setup()
    ctx.compute_level_populations(True, 2, "max", "fp32")
    P = ctx.populations()
    ctx.close()
    return P


def test_on_request():
    P = _solve()
    before = _free()
    kept = hip.release_memory()
    print(f"\n[memory] {kept} bytes kept by a closed context", flush=True)
    assert 100e6 < kept <= 2 << 30
    assert _free() >= before + 0.9 * kept
    assert hip.release_memory() == 0
    assert np.array_equal(_solve(), P)


def test_an_allocation_that_does_not_fit_takes_it_back():
    """2^42 rows of the network's inputs fit no card: the call fails with an error,
    having given all kept memory back, and the library goes on."""
    P = _solve()
    net = hip.Mlp(seed=0)
    X = np.zeros((1, 8), np.float32)
    rc = net.lib.mgr_mlp_forward(net.h, X.ctypes.data_as(C.c_void_p), 1 << 42, X.ctypes.data_as(C.c_void_p))
    assert rc != 0
    assert hip.release_memory() == 0
    assert np.all(np.isfinite(net.forward(X)))
    net.close()
    assert np.array_equal(_solve(), P)
