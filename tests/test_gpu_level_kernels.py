"""The rate equations with eight lanes per cell (2 to 8 levels, 32 cells per
block; one thread per cell beyond) and J_eff from rows of J in LDS (up to 8
cells per block; one thread per cell and line where a row does not fit), each
at the edges of its range, against the oracle.  The systems are pivoted from
their first column on: the conservation row's ones are the largest entries.
Bars: FP64 field 1e-10, populations of one solve 1e-9, as in the parity tests.
"""
import numpy as np
import pytest

from magritte_amd.setup import synthetic
from oracle.py_oracle import Oracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return float(np.max(np.abs(a - b) / np.maximum(np.abs(b), 1e-300)))


# (cells per side, levels, roots): 27, 125 or 216 cells, none a multiple of 32
# or 8; bins from 1 to past a row's 48 KB (4010 bins and their indices)
@pytest.mark.parametrize("n,nlev,nquads", [(6, 2, 1), (5, 3, 7), (6, 4, 31), (5, 5, 31), (6, 6, 13), (5, 7, 101),
                                           (6, 8, 31), (5, 9, 7), (6, 10, 31), (3, 3, 2005)])
def test_jeff_and_rate_equations(n, nlev, nquads):
    from magritte_amd.hip import Context
    print(f"\n[levels] n {n}, {nlev} levels, {nquads} roots", flush=True)
    m = synthetic.envelope_model(n=n, seed=nlev, nside=1, nlev=nlev, nquads=nquads)
    orc, ctx = Oracle(m).setup(), Context(m).setup()
    orc.compute_radiation_field()
    orc.compute_Jeff()
    ctx.compute_radiation_field("fp64")
    ctx.compute_Jeff()
    Jl_g, Je_g, Jd_g = ctx.Jeff()
    Jl_o, Je_o, Jd_o = orc.Jeff()
    assert rel(Jl_g, Jl_o) < 1e-10
    scale = np.maximum(np.abs(Jl_o), np.abs(Jd_o))
    assert float(np.max(np.abs(Je_g - Je_o) / scale)) < 1e-10
    assert float(np.max(np.abs(Jd_g - Jd_o) / scale)) < 1e-10
    orc.update_using_statistical_equilibrium()
    orc.check_for_convergence()
    conv_g = ctx.compute_level_populations_from_stateq()
    assert rel(ctx.populations(), orc.populations()) < 1e-9
    fo = orc.convergence()
    assert conv_g[0] == pytest.approx(fo[0], rel=1e-9, abs=1e-12)
    assert conv_g[1] == pytest.approx(fo[1], rel=1e-6)
    assert conv_g[2] == pytest.approx(fo[2], rel=1e-6)


@pytest.mark.parametrize("n,nlev,nquads", [(5, 4, 31), (3, 3, 2005)])
def test_iteration_sums_lambda_in_the_same_order(n, nlev, nquads):
    """One iteration adds the waves' shares of Lambda* where it takes J_eff; the
    separate calls add them first: the same bits."""
    from magritte_amd.hip import Context
    m = synthetic.envelope_model(n=n, seed=1, nside=1, nlev=nlev, nquads=nquads)
    a, b = Context(m).setup(), Context(m).setup()
    a.ali_iteration(False, "fp32")
    b.compute_radiation_field("fp32")
    b.compute_Jeff()
    for x, y in zip(a.Jeff(), b.Jeff()):
        assert np.array_equal(x, y)
    assert np.array_equal(a.lambda_diag(), b.lambda_diag())
    b.compute_level_populations_from_stateq()
    assert np.array_equal(a.populations(), b.populations())
