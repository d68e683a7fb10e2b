"""GPU: the single-pass fold resolves the sizes and starts of
test_gpu_fold_units.py by itself.  A phase that it cannot resolve is replayed
serially behind it, with the same result, so equality with the serial fold
alone does not show that the single pass ran; the count of replays does."""
import pytest

from test_gpu_fold_units import STARTS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("backint", [False, True])
@pytest.mark.parametrize("starts", sorted(STARTS))
@pytest.mark.parametrize("N", [16, 66, 4094, 4096, 4098, 8194, 49154, 262144])
def test_no_phase_is_replayed(N, starts, backint):
    from emri_kludge_suite_amd import GPUAAK
    gamma, psi, alph = STARTS[starts]
    for s, M in ((0.5, 1e6), (0.9, 3e5)):
        print("case fold-single N=%d starts=%s backint=%d s=%g" % (N, starts, backint, s), flush=True)
        g = GPUAAK(1.0, max(1, N // 10), N, 100.0, 15.0, True, backint)
        g.set_nmax(4)
        g.gpu_gen_AAK(0.5, s, 9.0, 0.2, M, 10.0, gamma, psi, alph, 1.1, 4.0, 0.7, 5.0, 1.0)
        assert g.info()["fold_fallbacks"] == 0
        g.close()
