"""GPU: e, v, M and S of fast sources, whose knots lie a few samples apart, so
that a workgroup's share of samples is cut to the knots its LDS holds: equal
to the oracle's splines bit for bit, at lengths where the share would be one,
two and four rows of 256 samples."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu

PLUNGE = [0.5, 0.5818, 9.4211, 0.3929, 119708.4349, 13.4395, 4.9582, 0.2884, 0.8303, 1.5676, 4.4618, 1.3913, 0.2321,
          1.0]
FAST = [0.5, 0.5, 14.0, 0.2, 2.5e5, 20.0, 1.0, 2.0, 3.0, 1.1, 4.0, 0.7, 5.0, 1.0]


@pytest.mark.parametrize("pars", ["plunge", "fast"])
@pytest.mark.parametrize("N", [2 ** 18, 2 ** 18 + 2, 2 ** 19 + 2, 2 ** 20])
def test_splines_of_dense_knots(N, pars):
    from emri_kludge_suite_amd import GPUAAK
    print("case rates-knots N=%d %s" % (N, pars), flush=True)
    p = PLUNGE if pars == "plunge" else FAST
    ref = ol.o_aak_wave(p, length=N, dt=15.0, n_max=1, want_dense=True)
    g = GPUAAK(1.0, N // 10, N, 100.0, 15.0, True, False)
    g.set_nmax(1)
    g.gpu_gen_AAK(*p)
    d = g.dense_arrays()
    print("  knots %d" % g.info()["K"], flush=True)
    assert N / g.info()["K"] < 20
    for k in ("e", "v", "M", "S"):
        assert np.array_equal(d[k], ref["dense_" + k]), k
    g.close()
