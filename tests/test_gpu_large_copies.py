"""Large results are copied to the host in 2 MB chunks by several threads (from
4 MB on): every byte arrives, at sizes around the chunk and the threshold, into
fresh and used arrays, and when two threads read one context at once."""
import ctypes as C
import threading

import numpy as np
import pytest

from magritte_amd.setup import synthetic

pytestmark = pytest.mark.gpu


# J of n^3 cells and 39 bins: 0.07, 3.6, 4.2, 4.9 and 34 MB
@pytest.mark.parametrize("n", [6, 23, 24, 25, 48])
def test_every_byte(n):
    from magritte_amd.hip import Context
    print(f"\n[copies] J of {n}^3 x 39", flush=True)
    ctx = Context(synthetic.regular_grid_model(n=n)).setup()
    ctx.compute_radiation_field("fp32")
    J = ctx.J()
    assert np.all(np.isfinite(J)) and np.all(J > 0)
    used = np.full(J.size, np.nan)
    for _ in range(2):   # the second time into memory that is there
        assert ctx.lib.mgr_get_J(ctx.h, used.ctypes.data_as(C.c_void_p)) == 0
        assert np.array_equal(used.reshape(J.shape), J)
    # cell by cell: the grid is uniform, so mirrored cells have the same J up to rounding
    K = J.reshape(n, n, n, -1)
    assert np.allclose(K, K[::-1, ::-1, ::-1], rtol=1e-4)
    results = [None, None]
    def read(i):
        results[i] = ctx.J()
    th = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert np.array_equal(results[0], J) and np.array_equal(results[1], J)
    ctx.close()


def test_next_context_on_used_memory():
    """The trace's large arrays are kept for the next context: models that take
    over another one's memory, of other sizes, in both trace passes (walks too
    long to record are scanned again) and from two threads, give the bits they
    give alone."""
    from magritte_amd.hip import Context
    makes = [lambda: synthetic.envelope_model(n=20, seed=1), lambda: synthetic.stress_model(n=16, seed=2),
             lambda: synthetic.envelope_model(n=18, seed=3, nlev=4)]

    def solve(i, steps=-1):
        ctx = Context(makes[i]()).setup()
        ctx.set_trace_options(steps, True)
        ctx.trace()
        ctx.compute_level_populations(True, 6, "max", "fp32")
        out = ctx.populations(), ctx.J()
        ctx.close()
        return out

    alone = [solve(i) for i in range(3)]
    for i, steps in ((1, -1), (0, 4), (2, 0), (0, -1), (1, 4)):
        for a, b in zip(solve(i, steps), alone[i]):
            assert np.array_equal(a, b), i
    results = {}
    th = [threading.Thread(target=lambda i=i: results.update({i: solve(i)})) for i in range(3)]
    [t.start() for t in th]
    [t.join() for t in th]
    for i in range(3):
        for a, b in zip(results[i], alone[i]):
            assert np.array_equal(a, b), i
