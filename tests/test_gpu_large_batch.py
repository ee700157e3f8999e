"""A batch of more (cell, ray) entries than a launch has waves (2^32 / 64): the
far-end intensity cache covers every one.  350 copies of one small model with
48 rays, 68.8 million entries of one bin: every copy gets the bits of the
first, with the cache and without."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic

pytestmark = pytest.mark.gpu


def test_far_cache_of_a_large_batch():
    from magritte_amd.hip import BatchContext
    m = synthetic.envelope_model(n=16, nside=2, nlev=2, nquads=1, seed=5)
    K = 350
    assert K * m.ncells * m.nrays * 64 > 2 ** 32
    print(f"\n[large batch] {K} x {m.ncells} cells x {m.nrays} rays", flush=True)
    ctx = BatchContext([m] * K).setup()
    ctx.trace()
    fields = []
    for cache in (True, False):
        ctx.set_far_cache(cache)
        ctx.compute_radiation_field("fp32")
        J = ctx.J().reshape(K, -1)
        assert np.array_equal(J, np.broadcast_to(J[0], J.shape)), cache
        fields.append(J[0])
    assert np.array_equal(fields[0], fields[1])
    ctx.close()
