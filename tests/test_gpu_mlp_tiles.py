"""GPU: the network's gradient at the edges of its tiles (32 rows) and of its
grid (256 workgroups, then several tiles each).  The bound is that of
test_gpu_mlp.py: a BF16 rounding tie decided differently in FP32 and FP64 moves
one element by 2^-8, all else is FP32 summation (1e-5)."""
import numpy as np
import pytest

import mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 31, 32, 33, 65, 8191, 8193, 24580])
def test_gradient_at_tile_edges(n):
    from emri_kludge_suite_amd.freqmap_mlp import FreqMapModel
    rng = np.random.default_rng(1000 + n)
    p = rng.normal(0, 0.15, R.NP)
    for name in ("W2", "W3", "W4"):
        o, k = R.OFF[name]
        p[o:o + k] = rng.normal(0, np.sqrt(2.0 / R.H), k)
    p = p.astype(np.float32).astype(np.float64)
    X = rng.normal(size=(n, 4)).astype(np.float32)
    T = rng.normal(size=(n, 3)).astype(np.float32)
    print("case mlp gradient n=%d" % n, flush=True)
    m = FreqMapModel(0)
    m.set(p.astype(np.float32), None)
    m.gradient(X[: n // 2 + 1] + 1, T[: n // 2 + 1])  # another size first: its scratch does not reach the next
    g, loss = m.gradient(X, T)
    ref_loss, ref = R.loss_and_grad(p, X.astype(np.float64), T.astype(np.float64), bf=True)
    assert loss == pytest.approx(ref_loss, rel=1e-5)
    for name, (o, k) in R.OFF.items():
        rel = np.linalg.norm(g[o:o + k].astype(np.float64) - ref[o:o + k]) / np.linalg.norm(ref[o:o + k])
        print("  %s rel L2 %.3e" % (name, rel), flush=True)
        assert rel < 2e-3, name
