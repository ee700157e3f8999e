"""The band kernel's walk of a ray pair at its edges: rays of more points than
a window (32) and more steps than a batch (64 lanes), one bin to more than two
chunks of bins, one and several lines per bin, lanes in either order, bands of
1 to 7 off-diagonals, pairs shorter than the band.  Passing over the
out-of-window points must not change a bit, and the elements meet the
oracle's at the band tests' bar (1e-10)."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic
from oracle.py_oracle import Oracle

pytestmark = pytest.mark.gpu


def _long(n=70):
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


MODELS = {
    "envelope6": lambda: synthetic.envelope_model(n=6, seed=2, nside=1),
    "stress5": lambda: synthetic.stress_model(n=5, seed=3, nside=1),
    "long70": _long,
    "one_bin": lambda: synthetic.regular_grid_model(n=4, nquads=1),
    "blended5": lambda: synthetic.blended_model(n=5, seed=6, nside=1, nquads=17),
}


@pytest.mark.parametrize("name,n_off_diag", [("envelope6", 2), ("envelope6", 8), ("stress5", 2), ("long70", 2),
                                             ("long70", 8), ("one_bin", 4), ("blended5", 3)])
def test_windows_and_oracle(name, n_off_diag):
    from magritte_amd.hip import Context
    print(f"\n[band windows] {name} n_off_diag {n_off_diag}", flush=True)
    m = MODELS[name]()
    m.n_off_diag = n_off_diag
    orc, ctx = Oracle(m).setup(), Context(m).setup()
    orc.compute_radiation_field()
    ctx.compute_radiation_field("fp64")
    cells, L = ctx.lambda_band_raw()
    band_o = orc.lambda_band()
    band_g, _ = ctx.lambda_band()
    worst = 0.0
    for p in range(orc.N):
        for k in range(orc.L):
            e, g = dict(band_o[p][k]), band_g.get((p, k), {})
            assert set(e) == set(g), (p, k)
            for nr, v in e.items():
                worst = max(worst, abs(g[nr] - v) / max(abs(v), 1e-300))
    print(f"[band windows] max rel err {worst:.3e}", flush=True)
    assert worst < 1e-10
    ctx.set_window_skip(False)
    ctx.compute_radiation_field("fp64")
    cells2, L2 = ctx.lambda_band_raw()
    assert np.array_equal(cells, cells2)
    assert np.array_equal(L[cells >= 0], L2[cells2 >= 0])
