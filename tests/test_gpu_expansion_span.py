"""GPU: FP64 mode sums with one expansion per 1024 samples (the default from
2^18 samples on) against one per 256: just below and at the line, a year, a
source that plunges (blocks expanded again per 256 samples, and summed per
sample), and lengths that leave part blocks.  Either order bound is 1e-17 per
amplitude; 1e-12 is what the rounding of up to 60 harmonics of some thousand
radians leaves between the two expansions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CALM = [0.5, 0.5, 9.0, 0.2, 1e6, 10.0, 1.0, 2.0, 3.0, 1.1, 4.0, 0.7, 5.0, 1.0]
PLUNGE = [0.5, 0.5818, 9.4211, 0.3929, 119708.4349, 13.4395, 4.9582, 0.2884, 0.8303, 1.5676, 4.4618, 1.3913, 0.2321,
          1.0]


@pytest.mark.parametrize("pars", ["calm", "plunge"])
@pytest.mark.parametrize("N,shift", [(258, 0), (2 ** 18 - 2, 0), (2 ** 18, 2), (2 ** 18 + 258, 2), (2 ** 21, 2)])
def test_wide_expansions_agree_with_narrow_ones(N, shift, pars):
    from emri_kludge_suite_amd import GPUAAK
    print("case expansion-span N=%d %s" % (N, pars), flush=True)
    g = GPUAAK(1.0, max(1, N // 10), N, 100.0, 15.0, True, False)
    g.set_nmax(50)
    out = {}
    for xs in (-2, 0, 2):
        g.set_tuning(exp_shift=xs)
        g.gpu_gen_AAK(*(CALM if pars == "calm" else PLUNGE))
        t, hI, hII = g.GetWaveform()
        out[xs] = np.stack([hI, hII])
    g.close()
    assert np.array_equal(out[-2], out[shift])  # the default's line
    rel = np.linalg.norm(out[2] - out[0]) / np.linalg.norm(out[0])
    print("  rel L2 of 1024 against 256 samples: %.2e" % rel, flush=True)
    assert np.linalg.norm(out[0]) > 0 and rel <= 1e-12
