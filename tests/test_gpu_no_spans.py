"""Without the spans of sub-points (set_window_skip(spans=False), as where there
is no memory for them) the field and band kernels pass over whole steps by their
out-of-window bits: the same bits of J, Lambda* and its bands, and still less
time than evaluating every point."""
import numpy as np
import pytest

from magritte_amd.setup import synthetic

pytestmark = pytest.mark.gpu

MODELS = {
    "envelope9": lambda: synthetic.envelope_model(n=9, seed=2, nside=1),
    "stress7": lambda: synthetic.stress_model(n=7, seed=3, nside=1),
    "bins402": lambda: synthetic.envelope_model(n=6, seed=5, nside=1, nquads=67),
    "blended7": lambda: synthetic.blended_model(n=7, seed=6, nside=1, nquads=17),
}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", list(MODELS))
def test_same_bits(name, precision):
    from magritte_amd.hip import Context
    print(f"\n[no spans] {name} {precision}", flush=True)
    m = MODELS[name]()
    if name == "envelope9":
        m.n_off_diag = 2
    ctx = Context(m).setup()
    out = []
    for enable, spans in ((False, True), (True, False), (True, True)):
        ctx.set_window_skip(enable, spans)
        ctx.compute_radiation_field(precision)
        out.append([ctx.J(), ctx.lambda_diag()] + ([ctx.lambda_band_raw()[1]] if m.n_off_diag == 2 else []))
    for got in out[1:]:
        for a, b in zip(got, out[0]):
            assert np.array_equal(a, b)
    ctx.close()


def test_whole_steps_are_passed_over():
    """Most steps of a fast wind are out of every window: without spans the FP64
    kernel takes well under the time of evaluating all of their points."""
    from magritte_amd.hip import Context
    ctx = Context(synthetic.envelope_model(n=24, nside=1, v_inf=60e3)).setup()
    ms = {}
    for enable, spans in ((False, True), (True, False)):
        ctx.set_window_skip(enable, spans)
        times = []
        for _ in range(6):
            ctx.compute_radiation_field("fp64")
            times.append(ctx.last_radiation_field_ms())
        ms[enable] = min(times[1:])
    print(f"\n[no spans] every point {ms[False]:.3f} ms, whole steps passed over {ms[True]:.3f} ms", flush=True)
    assert ms[True] < 0.8 * ms[False]
    ctx.close()
