"""CPU: which transform the inner-product stage takes at a length.  Lengths
whose half is a product of primes up to 17 need no convolution in rocFFT, whose
radices end there, and stay with it; so do those below 64 samples.  The others
take the convolution, whose factors must hold 2M - 1 points."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def form():
    from emri_kludge_suite_amd import _lib

    def f(n):
        R, Cc = np.zeros(1, dtype=np.int32), np.zeros(1, dtype=np.int32)
        return _lib.lib().aak_test_transform(n, _lib.iptr(R), _lib.iptr(Cc)), int(R[0]), int(Cc[0])
    return f


def _smooth(m):
    for q in (2, 3, 5, 7, 11, 13, 17):
        while m % q == 0:
            m //= q
    return m == 1


def test_lengths_that_the_library_takes_without_a_convolution(form, monkeypatch):
    monkeypatch.delenv("AAK_FFT", raising=False)
    for n in (34, 38, 46, 62, 1088, 1156, 8704, 278528, 344250, 2000000, 2228224, 2263040, 4718592, 4718594, 8388610):
        assert form(n) == (0, 0, 0), n


def test_every_length_keeps_the_rule(form, monkeypatch):
    monkeypatch.delenv("AAK_FFT", raising=False)
    rng = np.random.default_rng(3)
    lengths = list(range(16, 20000, 2)) + (2 * rng.integers(10000, 2359296, 20000)).tolist() + [4194302, 4194306, 4718590]
    for n in lengths:
        kind, R, Cc = form(n)
        if n >= 256 and n & (n - 1) == 0:
            assert kind == 1 and R * Cc == n // 2
        elif n < 64 or _smooth(n // 2):
            assert kind == 0
        else:
            assert kind == 2 and R * Cc >= n - 1, n
            if n >= 514:
                assert 2 * R * Cc < 3 * (n - 1), n
            if n >= 1538:
                assert 3 * R * Cc < 4 * n, n


def test_the_library_for_every_length(form, monkeypatch):
    monkeypatch.setenv("AAK_FFT", "rocfft")
    for n in (256, 2103840, 1 << 21, 4002):
        assert form(n) == (0, 0, 0), n
