"""The FP32 field kernel of staged steps (k_field_staged) and when it runs: models
of many lines or bins, dark boundaries, very long steps and the skip switched off.
It gives the bits of the kernel that lays points out per lane, at every launch
shape, with scattering, in the iteration's graphs and in a batch, and meets the
oracle at the parity bar (1e-5 of the largest J)."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic
from oracle.py_oracle import Oracle

pytestmark = pytest.mark.gpu

POINTS, STAGED = "k_radiation_field<float", "k_field_staged"


def _cold(m, T):
    m.boundary_temperature = np.full(m.nboundary, T)
    return m


def _envelope(n, seed, **kw):
    return synthetic.envelope_model(n=n, seed=seed, nside=1, **kw)


# model, the kernel that runs it with the skip on
MODELS = {
    "plain": (lambda: _envelope(8, 2), POINTS),
    "13 lines": (lambda: _envelope(6, 3, nlev=14, nquads=9), POINTS),
    "15 lines": (lambda: _envelope(6, 3, nlev=16, nquads=9), STAGED),
    "31 lines": (lambda: _envelope(6, 4, nlev=32, nquads=7), STAGED),
    "31 lines, jumps": (lambda: synthetic.stress_model(n=5, seed=5, nside=1, nlev=32, nquads=13), STAGED),
    "16 chunks": (lambda: _envelope(5, 6, nquads=170), POINTS),
    "17 chunks": (lambda: _envelope(5, 6, nquads=171), STAGED),
    "12 lines, 6 chunks": (lambda: _envelope(6, 6, nlev=13, nquads=27), STAGED),
    "several lines a bin": (lambda: synthetic.blended_model(n=6, seed=7, nside=1, nquads=17), POINTS),
    "several lines a bin, 6 chunks": (lambda: synthetic.blended_model(n=6, seed=7, nside=1, nquads=33), STAGED),
    "boundary at 2.6 K": (lambda: _cold(_envelope(8, 8), 2.6), POINTS),
    "boundary at 2 K": (lambda: _cold(_envelope(8, 8), 2.0), STAGED),
    "boundary at 0.05 K": (lambda: _cold(_envelope(8, 8), 0.05), STAGED),
}


def _context(m):
    from magritte_amd.hip import Context
    ctx = Context(m).setup()
    if m.boundary_temperature is not None:
        ctx.compute_boundary_intensities(m.boundary_temperature)
    return ctx


def _field(ctx, precision="fp32"):
    ctx.compute_radiation_field(precision)
    return ctx.J(), ctx.lambda_diag()


@pytest.mark.parametrize("name", list(MODELS))
def test_kernel_bits_and_oracle(name):
    make, kernel = MODELS[name]
    print(f"\n[staged] {name}", flush=True)
    m = make()
    ctx = _context(m)
    J, L = _field(ctx)
    assert ctx.last_radiation_field_kernel().startswith(kernel)
    orc = Oracle(m).setup()
    if m.boundary_temperature is not None:
        orc.compute_boundary_intensities(m.boundary_temperature)
    orc.compute_radiation_field()
    assert np.max(np.abs(J - orc.J())) <= 1e-5 * np.max(orc.J())
    for enable, spans in ((True, False), (False, True)):   # with the steps' bits and without
        ctx.set_window_skip(enable, spans)
        for shape in ((1, 2), (1, 16), (2, 31), (3, 32), (4, 33)):
            ctx.set_radiation_field_shape("fp32", *shape)
            J1, L1 = _field(ctx)
            assert ctx.last_radiation_field_kernel().startswith(STAGED)
            assert ctx.radiation_field_shape("fp32")[0] == shape
            assert np.array_equal(J1, J) and np.array_equal(L1, L), (enable, spans, shape)
    ctx.close()


@pytest.mark.parametrize("side,kernel", [(1e17, POINTS), (2e18, POINTS), (1e20, STAGED)])
def test_long_steps(side, kernel):
    """Cells of up to 1e19 m: y leaves the range in which runs can be passed over at
    some points (2e18 m: above 6 to 9) or everywhere (1e20 m)."""
    print(f"\n[staged] box of {side:g} m", flush=True)
    for model in (_envelope(9, 9, side=side, n0=1e29 / side),
                  synthetic.stress_model(n=7, seed=9, nside=1, side=side, n0=1e31 / side)):
        ctx = _context(model)
        J, L = _field(ctx)
        assert ctx.last_radiation_field_kernel().startswith(kernel)
        for enable, spans in ((True, False), (False, True)):
            ctx.set_window_skip(enable, spans)
            J1, L1 = _field(ctx)
            assert np.array_equal(J1, J) and np.array_equal(L1, L)
        ctx.close()


def test_scattering():
    ctx = _context(_envelope(7, 10))
    ctx.set_scattering(True)
    _field(ctx)
    u = ctx.u()
    ctx.set_window_skip(True, spans=False)
    _field(ctx)
    assert ctx.last_radiation_field_kernel().startswith(STAGED)
    assert np.array_equal(ctx.u(), u)
    ctx.close()


def test_graphs_follow_the_boundary():
    """The iteration's graphs hold a kernel: a boundary that turns dark, and bright
    again, gives what a new context gives."""
    m = _envelope(8, 11)
    ctx = _context(m)
    P = ctx.populations()
    for T in (2.72548, 0.5, 2.72548):
        ctx.compute_boundary_intensities(np.full(m.nboundary, T))
        ctx.set_populations(P)
        ctx.ali_iteration(False, "fp32")
        assert ctx.last_radiation_field_kernel().startswith(STAGED if T < 1 else POINTS)
        new = _context(m)
        new.compute_boundary_intensities(np.full(m.nboundary, T))
        new.ali_iteration(False, "fp32")
        assert np.array_equal(ctx.J(), new.J()) and np.array_equal(ctx.populations(), new.populations())
        new.close()
    ctx.close()


def test_batch():
    """Models of a batch that converge at different iterations, by staged steps."""
    from magritte_amd.hip import BatchContext
    models = [_envelope(n, n, nlev=17, nquads=9, n0=10.0 ** e) for n, e in ((5, 12), (7, 14), (4, 10))]
    batch = BatchContext(models).setup()
    batch.compute_level_populations(True, 20, "fraction", "fp32")
    assert batch.last_radiation_field_kernel().startswith(STAGED)
    its, _ = batch.convergence()
    for m, P, n in zip(models, batch.split(batch.populations()), its):
        ctx = _context(m)
        assert ctx.compute_level_populations(True, 20, "fraction", "fp32") == n
        assert np.array_equal(ctx.populations(), P)
        ctx.close()
    batch.close()
