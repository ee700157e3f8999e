"""The network's kernels at the edges of their tiles: 16 rows per wave, 64 per
workgroup and at most 256 workgroups of the gradient, with normalised inputs
and targets, against the CPU reference at the bars of test_gpu_mlp (loss 1e-4,
gradient blocks 3e-2 in relative L2 norm, outputs 1e-2 of the largest)."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 16384, 16385, 16449])
def test_tiles_match_reference(n):
    from magritte_amd.hip import Mlp
    print(f"\n[mlp tiles] n={n}", flush=True)
    rng = np.random.default_rng(300 + n)
    p = {"W1": rng.normal(0, 0.3, (8, 128)), "b1": rng.normal(0, 0.1, 128),
         "W2": rng.normal(0, 0.075, (128, 128)), "b2": rng.normal(0, 0.1, 128),
         "W3": rng.normal(0, 0.075, (128, 7)), "b3": rng.normal(0, 0.1, 7)}
    p = {k: np.asarray(v, np.float32).astype(np.float64) for k, v in p.items()}
    xm, xs = rng.normal(0, 1, 8).astype(np.float32), rng.uniform(0.5, 2, 8).astype(np.float32)
    ym, ys = rng.normal(0, 1, 7).astype(np.float32), rng.uniform(0.5, 2, 7).astype(np.float32)
    net = Mlp(seed=1)
    net.set_params(p)
    net.set_normalisation(xm, xs, ym, ys)
    X = rng.normal(0, 1, (n, 8)).astype(np.float32)
    T = rng.normal(0, 1, (n, 7)).astype(np.float32)
    Xn = (X.astype(np.float64) - xm) / xs
    Tn = (T.astype(np.float64) - ym) / ys
    loss, g = net.loss_grad(X, T)
    lo, go = mo.loss_and_grads(p, Xn, Tn)
    assert abs(loss - lo) <= 1e-4 * lo
    for k in go:
        err = np.linalg.norm(g[k] - go[k]) / np.linalg.norm(go[k])
        assert err < 3e-2, (k, err)
    Y = net.forward(X)
    Yo, _ = mo.forward(p, Xn)
    Yo = Yo * ys + ym
    assert np.abs(Y - Yo).max() / np.abs(Yo).max() < 1e-2
    net.close()
