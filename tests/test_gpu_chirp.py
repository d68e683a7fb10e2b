"""GPU: the inner-product stage at lengths whose half has a prime factor above
13, as a cyclic convolution (Bluestein) on the library's own FFT: every side of
the convolution (columns 2^a, rows 2^a, 3 2^a and 9 2^a), the longest length
of a product and the shortest of the next, the smallest and largest taken, and
a length of one year at 15 s.  The reference is numpy's pocketfft; the bounds
are 1e-13 relative, about fifty times the rounding of two chained transforms of
2^22 points (eps log2 L) and a tenth of the bound of the other lengths' test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [34, 254, 258, 766, 1022, 1534, 2046, 2050, 2302, 3070, 4606, 6142, 9214, 9218, 12286,
                               16382, 24574, 36862, 49150, 65534, 65538, 73726, 147454, 196606, 294910, 524290, 589822,
                               786430, 1048574, 1179646, 1572862, 2097150, 2097154, 2103840, 2359298, 3145726,
                               4194302])
def test_inner_product_of_any_even_length(N, monkeypatch):
    from emri_kludge_suite_amd import GPUAAK
    monkeypatch.delenv("AAK_FFT", raising=False)
    print("case chirp N=%d" % N, flush=True)
    rng = np.random.default_rng(N)
    nb = N // 2 + 1
    h = rng.standard_normal((2, N))
    w = rng.uniform(0.5, 2.0, (2, nb))
    d = (rng.standard_normal((2, nb)) + 1j * rng.standard_normal((2, nb))) * w
    g = GPUAAK(1.0, max(N // 10, 16), N, 100.0, 10.0, True, False)
    g.input_data(d[0], d[1], w[0], w[1])
    H = np.fft.rfft(h, axis=1) * w
    dh, hh = 4.0 * np.sum(np.real(np.conj(H) * d)), 4.0 * np.sum(np.abs(H) ** 2)
    for _ in range(2):  # the scratch of the first pass does not reach the second
        (a, b), spec, fused = g.inner_product_stage(h[0], h[1])
        err = float(np.sqrt(np.sum(np.abs(spec - H) ** 2) / np.sum(np.abs(H) ** 2)))
        print("  dh err %.2g hh err %.2g spectrum %.2g" % (abs(a - dh) / hh, abs(b - hh) / hh, err), flush=True)
        assert not fused
        assert err <= 1e-13 and abs(a - dh) <= 1e-13 * hh and abs(b - hh) <= 1e-13 * hh
    g.close()
