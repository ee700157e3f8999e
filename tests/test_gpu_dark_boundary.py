"""Behind a boundary without radiation the lines' far wings are all there is:
a bin whose window (11 widths) holds no line at any point has an intensity of
exactly 0, as the reference's.  The last line's upper wing is set apart: the
reference's window has no upper end there, and passing over points has one (such
a wing is below 3e-53 of the line's opacity).  FP64 meets the oracle to 1e-10 of
each J above 1e-200 (profile arguments of up to 450 in the exponent, 3e-13; the
oracle's unscaled values underflow further out), FP32 to 1e-5 of the largest J.
Passing over points gives the same bits."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic
from oracle.py_oracle import Oracle

pytestmark = pytest.mark.gpu


def _wide(m, scale):
    m.roots = m.roots * scale
    return m


MODELS = {
    # roots of up to 30 widths in a static model, 12 and 28 in moving ones
    "regular": lambda: _wide(synthetic.regular_grid_model(n=6, nquads=41), 6.0),
    "envelope": lambda: _wide(synthetic.envelope_model(n=6, seed=8, nside=1, nquads=31, v_inf=1e3), 5.6),
    "bins over five chunks": lambda: _wide(synthetic.envelope_model(n=5, seed=9, nside=1, nquads=81, v_inf=1e3), 5.6),
    "two lines a bin": lambda: _wide(synthetic.blended_model(n=6, seed=6, nside=1, nquads=21, v_inf=1e3), 5.6),
}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", list(MODELS))
def test_nothing_beyond_the_window(name, precision):
    from magritte_amd.hip import Context
    print(f"\n[dark] {name} {precision}", flush=True)
    m = MODELS[name]()
    orc, ctx = Oracle(m).setup(), Context(m).setup()
    cold = np.full(m.nboundary, 1e-3)
    orc.compute_boundary_intensities(cold)
    ctx.compute_boundary_intensities(cold)
    assert np.all(ctx.boundary_intensities() == 0.0)
    orc.compute_radiation_field()
    Jo = orc.J()
    inner = ctx.frequencies()[0] < m.linedata.frequency.max()   # not that wing
    assert np.any(Jo[inner] == 0.0) and np.any(Jo[~inner] > 0.0)
    for skip in (True, False):
        ctx.set_window_skip(skip)
        ctx.compute_radiation_field(precision)
        J = ctx.J()
        assert np.all(J[inner & (Jo == 0.0)] == 0.0), skip
        if precision == "fp64":
            held = (Jo > 1e-200) & inner if skip else Jo > 1e-200
            assert np.max(np.abs(J[held] / Jo[held] - 1)) < 1e-10, skip
        else:
            assert np.max(np.abs(J - Jo)) < 1e-5 * np.max(Jo), skip
        if skip:
            J_on, L_on = J, ctx.lambda_diag()
    assert np.array_equal(J[inner], J_on[inner]) and np.array_equal(ctx.lambda_diag(), L_on)
    if precision == "fp32":
        assert np.array_equal(J, J_on)
    ctx.close()
