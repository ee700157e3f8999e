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
