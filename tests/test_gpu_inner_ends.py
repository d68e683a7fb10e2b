"""GPU: aak_inner_product_noalloc with values at the first and the last bin
that are not finite.  The spectra of real series are real there, and their
product with the data is the complex one: an imaginary part of the data that is
not finite makes <h|d> NaN (0 times it), in the one-workgroup form, in the
four-step form and in the handle's likelihood stage alike, and leaves <h|h>."""
import numpy as np
import pytest

from test_zz_no_alloc import _case, _Hip, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("channel", [0, 1])
@pytest.mark.parametrize("N", [256, 8192, 16384])
def test_imaginary_parts_at_the_ends(N, channel, bad):
    from emri_kludge_suite_amd import GPUAAK, _lib
    f, hip = _noalloc(_lib), _Hip()
    g = GPUAAK(1.0, N // 10, N, 100.0, 10.0, True, False)
    try:
        for k in (0, N // 2):
            print("case inner-ends N=%d bin=%d" % (N, k), flush=True)
            hI, hII, dI, dII, w1, w2 = case = _case(np.random.default_rng(N), N)
            d = (dI, dII)[channel]
            d[k] = complex(d[k].real, bad)
            dev = [hip.upload(x) for x in case]
            out = hip.upload(np.zeros(2))
            assert hip.h.hipDeviceSynchronize() == 0
            assert f(*dev, N, out, None) == 0, _lib.last_error()
            dh, hh = hip.download(out, 2)
            g.input_data(dI, dII, w1, w2)
            (dh0, hh0), _, _ = g.inner_product_stage(hI, hII)
            assert np.isnan(dh0) and np.isnan(dh)
            assert np.isfinite(hh) and abs(hh - hh0) <= 1e-13 * hh0
    finally:
        hip.free()
        g.close()
