"""Forced launch shapes at the edge of a workgroup's LDS: with many lines and
waves the windows are shrunk to what fits 64 KB (rounding each wave's share up to
64 bytes once took these over it), and J and Lambda* keep the bits of the smallest
shape."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic

pytestmark = pytest.mark.gpu


# (levels, precision, waves, points): 7, 13, 35 and 37 lines
EDGES = [(8, "fp64", 4, 64), (14, "fp64", 4, 34), (14, "fp64", 4, 64), (36, "fp32", 3, 36), (36, "fp32", 3, 64),
         (38, "fp32", 3, 34)]


@pytest.mark.parametrize("nlev,precision,waves,points", EDGES)
def test_shapes_at_the_lds_limit(nlev, precision, waves, points):
    from magritte_amd.hip import Context
    print(f"\n[shapes] {nlev} levels {precision} {waves} waves {points} points", flush=True)
    ctx = Context(synthetic.envelope_model(n=5, seed=3, nside=1, nlev=nlev, nquads=11)).setup()
    ctx.set_radiation_field_shape(precision, 1, 2)
    ctx.compute_radiation_field(precision)
    J, Lam = ctx.J(), ctx.lambda_diag()
    ctx.set_radiation_field_shape(precision, waves, points)
    ctx.compute_radiation_field(precision)
    assert np.array_equal(ctx.J(), J) and np.array_equal(ctx.lambda_diag(), Lam)
    ctx.close()


@pytest.mark.parametrize("nlev,waves,points", [(8, 4, 64), (8, 4, 63), (14, 4, 34), (14, 2, 64), (36, 4, 32)])
def test_reported_shape_is_the_used_one(nlev, waves, points):
    """FP64 windows that do not fit are reported with the points they hold: as many
    as 64 KB have room for beside the line table, each wave's share (1792 bytes and
    32 per line of points + 1) in whole 64 bytes."""
    from magritte_amd.hip import Context
    ctx = Context(synthetic.envelope_model(n=4, seed=3, nside=1, nlev=nlev, nquads=5)).setup()
    ctx.set_radiation_field_shape("fp64", waves, points)
    w, c = ctx.radiation_field_shape("fp64")[0]
    L = nlev - 1

    def lds(n):
        return -(-(1792 + 32 * L * (n + 1)) // 64) * 64 * waves + 8 * L

    assert w == waves and 2 <= c <= points
    assert lds(c) <= 65536 and (c == points or lds(c + 1) > 65536)
    ctx.compute_radiation_field("fp64")
    assert ctx.radiation_field_shape("fp64")[0] == (w, c)
    ctx.close()


@pytest.mark.parametrize("nlev,fit", [(8, 36), (21, 10), (32, 6)])
def test_the_tuner_tries_the_window_that_fits(nlev, fit):
    """The FP64 windows timed: 16 points and as many as four waves per SIMD have LDS
    for (a sixteenth of 160 KB in multiples of 1280 bytes each: 10240), fewer than
    16 and even with many lines."""
    from magritte_amd.hip import Context
    ctx = Context(synthetic.envelope_model(n=6, seed=3, nside=1, nlev=nlev, nquads=7)).setup()
    ctx.compute_radiation_field("fp64")
    tried = {c for w, c, _ in ctx.radiation_field_shape("fp64")[1] if w == 1}
    assert {16, fit} <= tried
    assert ctx.radiation_field_shape("fp64")[0][1] in tried
    ctx.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_the_shape_outlives_the_frequencies(precision):
    """A tuned shape is reported, and used again, after the frequencies are set anew."""
    from magritte_amd.hip import Context
    ctx = Context(synthetic.envelope_model(n=7, seed=3, nside=1)).setup()
    ctx.compute_radiation_field(precision)
    tuned, J = ctx.radiation_field_shape(precision)[0], ctx.J()
    assert tuned[0] > 0
    ctx.compute_spectral_discretisation()
    assert ctx.radiation_field_shape(precision)[0] == tuned
    ctx.compute_boundary_intensities()
    ctx.compute_radiation_field(precision)
    assert ctx.radiation_field_shape(precision)[0] == tuned and np.array_equal(ctx.J(), J)
    ctx.close()
