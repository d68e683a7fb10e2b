"""GPU: aak_inner_product_noalloc at every length it takes: one workgroup up to
N = 8192, the four-step passes with the second one reading data and weights in
bin order beyond.  Against numpy's pocketfft; the bound, 1e-13 of <h|h>, is
that of the other lengths' test (fifty times the rounding of a transform of
2^20 points).  Two calls in a row, with other series, give each its own sums."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import _case, _Hip, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1 << k for k in range(8, 22)])
def test_inner_product_in_bin_order(N):
    from emri_kludge_suite_amd import _lib
    print("case inner-orders N=%d" % N, flush=True)
    f, hip = _noalloc(_lib), _Hip()
    try:
        for seed in (N, N + 1):
            hI, hII, dI, dII, w1, w2 = case = _case(np.random.default_rng(seed), N)
            dev = [hip.upload(x) for x in case]
            out = hip.upload(np.full(2, np.nan))
            assert hip.h.hipDeviceSynchronize() == 0
            assert f(*dev, N, out, None) == 0, _lib.last_error()
            dh, hh = hip.download(out, 2)
            H = [np.fft.rfft(h) * w for h, w in ((hI, w1), (hII, w2))]
            rh = 4.0 * sum(np.sum(np.abs(x) ** 2) for x in H)
            rd = 4.0 * sum(np.sum(np.real(np.conj(x) * d)) for x, d in zip(H, (dI, dII)))
            print("  dh err %.2g hh err %.2g" % (abs(dh - rd) / rh, abs(hh - rh) / rh), flush=True)
            assert abs(dh - rd) <= 1e-13 * rh and abs(hh - rh) <= 1e-13 * rh
    finally:
        hip.free()
