"""GPU: gradient calls about the line where their rows stop going through pinned
memory (16384 rows), against the float64 reference, and a short call after a
long one.  The bound is that of test_gpu_mlp.py (a BF16 rounding tie)."""
import numpy as np
import pytest

import mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16383, 16384, 16385])
def test_gradient_about_the_pinned_line(n):
    from emri_kludge_suite_amd.freqmap_mlp import FreqMapModel
    rng = np.random.default_rng(n)
    p = rng.normal(0, 0.15, R.NP)
    for name in ("W2", "W3", "W4"):
        o, k = R.OFF[name]
        p[o:o + k] = rng.normal(0, np.sqrt(2.0 / R.H), k)
    p = p.astype(np.float32).astype(np.float64)
    X = rng.normal(size=(n, 4)).astype(np.float32)
    T = rng.normal(size=(n, 3)).astype(np.float32)
    m = FreqMapModel(0)
    m.set(p.astype(np.float32), None)
    for rows in (n, 40):
        print("case mlp pinned rows=%d" % rows, flush=True)
        g, loss = m.gradient(X[:rows], T[:rows])
        ref_loss, ref = R.loss_and_grad(p, X[:rows].astype(np.float64), T[:rows].astype(np.float64), bf=True)
        assert loss == pytest.approx(ref_loss, rel=1e-5)
        for name, (o, k) in R.OFF.items():
            rel = np.linalg.norm(g[o:o + k].astype(np.float64) - ref[o:o + k]) / np.linalg.norm(ref[o:o + k])
            assert rel < 2e-3, name
