"""The image kernels' walk at its edges: rays of more points than a window (32)
and more steps than a batch (64 lanes), one bin to more than a chunk of bins,
several lines per bin, empty rays (boundary origins), against the oracle at the
image tests' bars (FP64 1e-10; FP32 2e-5 of |I| + 2 I_bdy)."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic
from oracle.py_oracle import Oracle

pytestmark = pytest.mark.gpu


def _long(n=70):
    """Four lines of n cells with rays along them only, up to n - 1 steps."""
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
    "long70": _long,
    "one_bin": lambda: synthetic.regular_grid_model(n=4, nquads=1),
    "stress6": lambda: synthetic.stress_model(n=6, seed=3, nside=1),
    "blended5": lambda: synthetic.blended_model(n=5, seed=6, nside=1, nquads=17),
}


@pytest.mark.parametrize("name", list(MODELS))
def test_windows_match_oracle(name):
    from magritte_amd.hip import Context
    m = MODELS[name]()
    orc, ctx = Oracle(m).setup(), Context(m)
    orc.compute_spectral_discretisation_image(3.0e-5)
    orc.compute_boundary_intensities()
    ctx.compute_spectral_discretisation_image(3.0e-5)
    ctx.compute_boundary_intensities()
    ctx.compute_LTE_level_populations()
    Ib2 = 2.0 * orc.boundary_intensities().max(axis=0)[None, :]
    for r in sorted({0, m.nrays // 2 - 1}):
        want = orc.compute_image(r)
        for prec, tol in (("fp64", 1e-10), ("fp32", 2e-5)):
            print(f"\n[image windows] {name} ray {r} {prec}", flush=True)
            for g, w in zip(ctx.compute_image(r, prec), want):
                den = np.abs(w) + (0.0 if prec == "fp64" else Ib2)
                assert float(np.max(np.abs(g - w) / np.maximum(den, 1e-300))) < tol
