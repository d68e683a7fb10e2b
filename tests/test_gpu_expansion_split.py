"""GPU: FP64 mode sums of sources that plunge slowly enough for only some of
their 1024-sample expansions to need an order above 8: these are expanded
again per 256 samples beside the wide ones.  The default span is 1024 samples
where the signal itself (not the grid) has 2^18 samples, else 256.  Wide and
narrow expansions then differ in rounding: by more than nothing, and by less
than 1e-12, what up to 60 harmonics of some thousand radians leave between two
expansions of order bound 1e-17 per amplitude."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ANGLES = [1.0, 2.0, 3.0, 1.1, 4.0, 0.7, 5.0, 1.0]
LONG = [0.5, 0.2655, 10.08, 0.414, 335500.0, 15.96] + ANGLES   # signal of 323 thousand samples at 15 s
SHORT = [0.5, 0.8568, 7.617, 0.1634, 323800.0, 15.76] + ANGLES  # 145 thousand


@pytest.mark.parametrize("N,pars,default", [(2 ** 19, LONG, 2), (2 ** 19, SHORT, 0), (2 ** 18, SHORT, 0),
                                            (2 ** 19 + 258, LONG, 2)])
def test_wide_and_split_expansions_mix(N, pars, default):
    from emri_kludge_suite_amd import GPUAAK
    print("case expansion-split N=%d default %d" % (N, default), flush=True)
    g = GPUAAK(1.0, N // 10, N, 100.0, 15.0, True, False)
    g.set_nmax(50)
    out, split = {}, {}
    for xs in (-2, 0, 2):
        g.set_tuning(exp_shift=xs)
        g.gpu_gen_AAK(*pars)
        info = g.info()
        out[xs] = np.stack(g.GetWaveform()[1:])
        split[xs] = info["split_blocks"]
    g.close()
    signal = info["i_plunge"] + info["i_buffer"]
    rel = np.linalg.norm(out[2] - out[0]) / np.linalg.norm(out[0])
    print("  signal %d, split %s, rel L2 of 1024 against 256 samples %.2e" % (signal, split, rel), flush=True)
    assert (signal >= 2 ** 18) == (default == 2) and signal < N
    assert split[0] == 0 and 0 < split[2] < signal // 1024
    assert split[-2] == split[default] and np.array_equal(out[-2], out[default])
    assert not np.array_equal(out[0], out[2])
    assert np.linalg.norm(out[0]) > 0 and rel <= 1e-12
