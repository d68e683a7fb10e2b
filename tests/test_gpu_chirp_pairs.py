"""GPU: the convolution at factors R x C that no other length of the tests
reaches, the shortest and the longest length it takes, and lengths with a
factor 17, which stay with rocFFT.  The reference is numpy's pocketfft; the
bounds are those of test_gpu_chirp.py, 1e-13 relative (about fifty times the
rounding of two chained transforms of 2^22 points)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _factors(N):
    from emri_kludge_suite_amd import _lib
    R, C = np.zeros(1, dtype=np.int32), np.zeros(1, dtype=np.int32)
    return _lib.lib().aak_test_transform(N, _lib.iptr(R), _lib.iptr(C)), (int(R[0]), int(C[0]))


@pytest.mark.parametrize("N,pair", [
    (74, (16, 16)), (4094, (64, 64)), (8188, (64, 128)), (18430, (128, 144)), (32766, (128, 256)), (98302, (256, 384)),
    (131070, (256, 512)), (262142, (512, 512)), (393214, (512, 768)), (524286, (512, 1024)), (4718590, (2048, 2304)),
    (34, None), (1156, None), (278528, None), (2228224, None)])
def test_inner_product_at_every_pair(N, pair, monkeypatch):
    from emri_kludge_suite_amd import GPUAAK
    monkeypatch.delenv("AAK_FFT", raising=False)
    print("case chirp-pairs N=%d" % N, flush=True)
    assert _factors(N) == ((2, pair) if pair else (0, (0, 0)))
    rng = np.random.default_rng(N)
    nb = N // 2 + 1
    h = rng.standard_normal((2, N))
    w = rng.uniform(0.5, 2.0, (2, nb))
    d = (rng.standard_normal((2, nb)) + 1j * rng.standard_normal((2, nb))) * w
    g = GPUAAK(1.0, max(N // 10, 16), N, 100.0, 10.0, True, False)
    g.input_data(d[0], d[1], w[0], w[1])
    H = np.fft.rfft(h, axis=1) * w
    dh, hh = 4.0 * np.sum(np.real(np.conj(H) * d)), 4.0 * np.sum(np.abs(H) ** 2)
    (a, b), spec, _ = g.inner_product_stage(h[0], h[1])
    err = float(np.sqrt(np.sum(np.abs(spec - H) ** 2) / np.sum(np.abs(H) ** 2)))
    print("  dh err %.2g hh err %.2g spectrum %.2g" % (abs(a - dh) / hh, abs(b - hh) / hh, err), flush=True)
    assert err <= 1e-13 and abs(a - dh) <= 1e-13 * hh and abs(b - hh) <= 1e-13 * hh
    g.close()
