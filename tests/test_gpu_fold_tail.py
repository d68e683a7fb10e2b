"""GPU: phases past the last folded step of a source that plunges.  They stay
at the value at the plunge (AAK.cc:265-269), also where the fold took the
serial replay, which runs behind the single pass: the dense phases after a
forced replay must be those of the single pass, bit for bit, to the last
sample."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLUNGE = [0.5, 0.5818, 9.4211, 0.3929, 119708.4349, 13.4395, 4.9582, 0.2884, 0.8303, 1.5676, 4.4618, 1.3913, 0.2321,
          1.0]
OTHER = [0.5, 0.5, 9.0, 0.2, 1e6, 10.0, 0.3, 0.4, 0.5, 1.1, 4.0, 0.7, 5.0, 1.0]


@pytest.mark.parametrize("replay", [1, 2])
@pytest.mark.parametrize("N,dt", [(8190, 600.0), (2 ** 17, 15.0)])
def test_tail_after_a_serial_replay(N, dt, replay):
    from emri_kludge_suite_amd import GPUAAK
    print("case fold-tail N=%d replay=%d" % (N, replay), flush=True)
    out = []
    for mode in (0, replay):
        g = GPUAAK(1.0, max(1, N // 10), N, 100.0, dt, True, False)
        g.set_nmax(4)
        g.gpu_gen_AAK(*OTHER)  # phases of another source in the buffers
        g.force_fold_replay(mode)
        g.gpu_gen_AAK(*PLUNGE)
        out.append((g.info(), g.dense_arrays()))
        g.close()
    (info, ref), (forced, got) = out
    last = info["i_plunge"] + info["i_buffer"]
    print("  last folded step %d, replays %d" % (last, forced["fold_fallbacks"]), flush=True)
    assert last < N - 100 and info["fold_fallbacks"] == 0 and forced["fold_fallbacks"] == 3
    for k in ("gim", "Phi", "alp"):
        assert np.all(ref[k][last + 2:] == ref[k][info["i_plunge"]]), k
        assert np.array_equal(got[k], ref[k]), k
