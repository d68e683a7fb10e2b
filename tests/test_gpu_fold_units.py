"""GPU: the single-pass fold on units of 64 steps, at the sizes and starts
where it can go wrong: part blocks, blocks of one step, the first block,
starts on and about powers of two, zero and negative starts, a phase that
crosses zero.  The serial replay adds the same increments one after another
in FP64 (AAK.cc:244-264), so the phases must be equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PHASES = ("gim", "Phi", "alp")
STARTS = {
    "plain": (1.0, 2.0, 3.0),
    "powers": (2.0, 0.0, 4.0),
    "zeros": (0.0, 0.0, 0.0),
    "negative": (-1.0, 3.0, -0.3),
    "below": (np.nextafter(8.0, 0), 6.0, np.nextafter(1.0, 0)),
}


@pytest.mark.parametrize("backint", [False, True])
@pytest.mark.parametrize("starts", sorted(STARTS))
@pytest.mark.parametrize("N", [16, 66, 4094, 4096, 4098, 8194, 49154, 262144])
def test_single_pass_fold_equals_the_serial_fold(N, starts, backint):
    from emri_kludge_suite_amd import GPUAAK
    gamma, psi, alph = STARTS[starts]
    for s, M in ((0.5, 1e6), (0.9, 3e5)):
        print("case fold-units N=%d starts=%s backint=%d s=%g" % (N, starts, backint, s), flush=True)
        pars = [0.5, s, 9.0, 0.2, M, 10.0, gamma, psi, alph, 1.1, 4.0, 0.7, 5.0, 1.0]
        g = GPUAAK(1.0, max(1, N // 10), N, 100.0, 15.0, True, backint)
        g.set_nmax(4)
        g.force_fold_replay(1)
        g.gpu_gen_AAK(*pars)
        ref = {k: v.copy() for k, v in g.dense_arrays().items() if k in PHASES}
        g.force_fold_replay(0)
        g.gpu_gen_AAK(*pars)
        got = g.dense_arrays()
        for k in PHASES:
            assert np.array_equal(got[k], ref[k]), (k, s)
        g.close()
