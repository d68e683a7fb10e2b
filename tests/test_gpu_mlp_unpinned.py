"""GPU: gradient calls where no pinned memory is to be had.  Their rows are
uploaded and read by the same kernels, so gradient and loss are those of the
pinned path bit for bit; a model may go from one path to the other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_gradient_without_pinned_memory():
    from emri_kludge_suite_amd import _lib
    from emri_kludge_suite_amd.freqmap_mlp import FreqMapModel
    m = FreqMapModel.load()
    for n in (1, 40, 4096, 16384):
        print("case mlp unpinned rows=%d" % n, flush=True)
        rng = np.random.default_rng(n)
        X, T = rng.normal(size=(n, 4)).astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32)
        res = []
        for off in (1, 0, 1):
            assert _lib.lib().aak_test_mlp_no_pinned(m._m, off) == 0
            res.append(m.gradient(X, T))
        for g, loss in res:
            assert np.linalg.norm(g) > 0 and np.array_equal(g, res[0][0]) and loss == res[0][1]
