"""The radiation-field kernels' windows, spans and runs at their edges.

A wave lays out the points of a ray pair from up to 63 steps at a time and
walks them in windows of `steps per chunk` points; out-of-window runs of points
are passed over, in the FP32 kernel only while the elimination's state passes
a test, otherwise with weaker assumptions or none.  Every way must give the
bits of evaluating every point (set_window_skip(False)) at every window size:
rays of more steps than a batch, steps of hundreds of sub-points, rays whose
boundary is dark (the test fails) or whose populations exceed the bound behind
the spans, one bin to more than five chunks of bins, one to ten lines per
bin's window.  J and the Lambda* diagonal also meet the oracle's at the bars
of the parity tests (1e-5 FP32, 1e-10 FP64)."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic
from oracle.py_oracle import Oracle

pytestmark = pytest.mark.gpu


def _long(n=150):
    """Four lines of n cells with rays along them only, up to n - 1 steps, and
    a velocity that swings through the windows."""
    m = synthetic.regular_grid_model(n=6, nquads=13)
    N = 4 * n
    q = np.arange(N)
    i, j, l = q % n, (q // n) % 2, q // (2 * n)
    m.position = np.stack([i, j, l], axis=1) * 1e13
    m.n_neighbors = np.where((i == 0) | (i == n - 1), 1, 2).astype(np.int64)
    m.neighbors = np.array([d for c in q for d in (c - 1, c + 1) if 0 <= c % n + d - c < n], np.int64)
    m.boundary2cell_nr = q[(i == 0) | (i == n - 1)].astype(np.int64)
    x = i / (n - 1.0)
    m.velocity = np.zeros((N, 3))
    m.velocity[:, 0] = 2e-5 * (x + 0.2 * np.sin(40 * x + j))
    m.rays, m.weights = np.array([[1.0, 0, 0], [-1.0, 0, 0]]), np.full(2, 0.5)
    m.temperature, m.vturb2 = np.full(N, 30.0), np.full(N, (150.0 / 2.99792458e8) ** 2)
    m.abundance = np.zeros((N, 3))
    m.abundance[:, 1], m.abundance[:, 2] = 1e8, 1e12
    return m


def _dark(m):
    m.boundary_temperature = np.full(m.nboundary, 0.05)
    return m


MODELS = {
    "envelope9": lambda: synthetic.envelope_model(n=9, seed=2, nside=1),
    "stress7": lambda: synthetic.stress_model(n=7, seed=3, nside=1),
    "long150": _long,
    "dark8": lambda: _dark(synthetic.envelope_model(n=8, seed=4, nside=1)),
    "one_bin": lambda: synthetic.regular_grid_model(n=6, nquads=1),
    "bins65": lambda: synthetic.regular_grid_model(n=5, nquads=65),
    "bins402": lambda: synthetic.envelope_model(n=6, seed=5, nside=1, nquads=67),
    "blended7": lambda: synthetic.blended_model(n=7, seed=6, nside=1, nquads=17),
}


@pytest.mark.parametrize("precision,tol", [("fp32", 1e-5), ("fp64", 1e-10)])
@pytest.mark.parametrize("name", list(MODELS))
def test_windows_and_runs(name, precision, tol):
    from magritte_amd.hip import Context
    print(f"\n[windows] {name} {precision}", flush=True)
    m = MODELS[name]()
    ctx = Context(m).setup()
    orc = Oracle(m).setup()
    if m.boundary_temperature is not None:
        ctx.compute_boundary_intensities(m.boundary_temperature)
        orc.compute_boundary_intensities(m.boundary_temperature)
    ctx.set_window_skip(False)
    ctx.compute_radiation_field(precision)
    J0, L0 = ctx.J(), ctx.lambda_diag()
    orc.compute_radiation_field()
    orc.compute_Jeff()
    J_o, L_o = orc.J(), orc.lambda_diag()
    assert np.max(np.abs(J0 - J_o)) <= tol * np.max(np.abs(J_o)) or np.max(np.abs(J0 / J_o - 1)) < tol
    assert np.max(np.abs(L0 - L_o)) <= tol * np.max(np.abs(L_o))
    ctx.set_window_skip(True)
    for shape in ((1, 2), (1, 5), (1, 16), (2, 31), (3, 32), (4, 63), (1, 64)):
        ctx.set_radiation_field_shape(precision, *shape)
        ctx.compute_radiation_field(precision)
        assert np.array_equal(ctx.J(), J0), shape
        assert np.array_equal(ctx.lambda_diag(), L0), shape
    ctx.close()


@pytest.mark.parametrize("scale", [0.5, 5.0, -3.0])
def test_populations_beyond_the_spans_bound(scale):
    """Populations of up to twice a cell's total are allowed for; larger ones,
    or negative ones, must not change what is evaluated."""
    from magritte_amd.hip import Context
    print(f"\n[windows] envelope8 populations x {scale}", flush=True)
    ctx = Context(synthetic.envelope_model(n=8, seed=7, nside=1)).setup()
    P = ctx.populations()
    P[::3] *= scale
    ctx.compute_radiation_field("fp32")   # spans built with the LTE populations
    ctx.set_populations(P)
    ctx.compute_radiation_field("fp32")
    J1, L1 = ctx.J(), ctx.lambda_diag()
    ctx.set_window_skip(False)
    ctx.compute_radiation_field("fp32")
    assert np.array_equal(ctx.J(), J1) and np.array_equal(ctx.lambda_diag(), L1)
    ctx.close()


@pytest.mark.parametrize("name", ["regular", "envelope"])
def test_fp64_bins_that_meet_no_line(name):
    """Roots up to 30 widths: the outer bins of a static model have no candidate
    line at any point, and the FP64 profile must still come out as exactly 0."""
    from magritte_amd.hip import Context
    m = (synthetic.regular_grid_model(n=6, nquads=41) if name == "regular" else
         synthetic.envelope_model(n=6, seed=8, nside=1, nquads=41))
    m.roots = m.roots * 6.0
    orc, ctx = Oracle(m).setup(), Context(m).setup()
    orc.compute_radiation_field()
    ctx.compute_radiation_field("fp64")
    J, Jo = ctx.J(), orc.J()
    assert np.all(np.isfinite(J))
    assert float(np.max(np.abs(J - Jo) / Jo)) < 1e-10
    assert np.all(np.isfinite(ctx.lambda_diag()))
