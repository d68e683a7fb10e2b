"""GPU: the phase rates at every sample against the same expressions in numpy
(one rounding per operation, AAK.cc:245-253): equal bit for bit, at lengths
about the workgroup's samples and the grid's sizes (256 samples per thread
row, 1024 workgroups), for light and heavy, near-circular, eccentric and
retrograde-leaning sources.  The divisions of the kernel share reciprocals, so
a wrong last bit would show here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _maps(v, e, Y, q):
    v2, e2, Y2, q2 = v * v, e * e, Y * Y, q * q
    v3, v4, e4 = v2 * v, v2 * v2, e2 * e2
    T = (2. * e4 * (240. + v2 * (-120. + v * (42. * (-27. + 4. * q2) * v + (-6567. + 1996. * q2) * v3 +
                                             48. * q * (8. + 77. * v2) * Y - 4. * q2 * v * (90. + 1577. * v2) * Y2))) +
         e4 * e2 * (560. + v2 * (-360. + 960. * q * v * Y + 8816. * q * v3 * Y +
                                 v4 * (-15565. + 24. * q2 * (200. - 629. * Y2)) +
                                 v2 * (-2742. + 80. * q2 * (5. - 11. * Y2)))) -
         8. * e2 * (-48. + v2 * (8. - 64. * q * v * Y - 688. * q * v3 * Y +
                                 2. * v2 * (99. + 16. * q2 * (-1. + 2. * Y2)) +
                                 v4 * (1233. + 8. * q2 * (-47. + 150. * Y2)))) +
         16. * (16. + v2 * (24. + v2 * (27. * (2. + 5. * v2) - 48. * q * v * Y +
                                        4. * q2 * (2. - v2 + (-2. + 3. * v2) * Y2))))) / (256. * v4)
    R = (16. + 8. * (-3. + e2) * v2 - 16. * (-3. + e2) * q * v3 * Y +
         8. * (33. + 4. * e2 - 3. * e4) * q * v3 * v2 * Y +
         v3 * v3 * (-351. + 132. * q2 + e2 * (-135. + 21. * e2 + 5. * e4 + 2. * (7. + e2) * q2) +
                    2. * (-204. + 13. * e2 * (-3. + e2)) * q2 * Y2) +
         2. * v2 * v2 * (-45. + 3. * e4 + 4. * q2 * (1. - 4. * Y2) + 2. * e2 * q2 * (1. + Y2))) / (16. * v)
    Th = (16. + 8. * (3. + e2) * v2 - 16. * (3. + e2) * q * v3 * Y -
          8. * (3. + e2) * (5. + 3. * e2) * q * v3 * v2 * Y +
          v3 * v3 * (135. - 54. * q2 + e2 * (5. * (27. + 9. * e2 + e4) + 2. * (-38. + e2) * q2) +
                     2. * (57. + 90. * e2 + 13. * e4) * q2 * Y2) +
          2. * v2 * v2 * (27. + 3. * e4 + 2. * q2 * (-1. + 7. * Y2) + 2. * e2 * (9. + q2 * (1. + Y2)))) / (16. * v)
    Ph = (16. + 8. * (3. + e2) * v2 - 16. * q * v3 * (-2. + (3. + e2) * Y) -
          8. * q * v3 * v2 * (-6. + 15. * Y + 3. * e4 * Y + 2. * e2 * (-4. + 7. * Y)) +
          2. * v2 * v2 * (27. + 3. * e4 + 2. * q2 * (-1. + Y) * (1. + 7. * Y) + 2. * e2 * (9. + q2 * (1. + Y2))) +
          v3 * v3 * (5. * e4 * e2 + e4 * (45. + q2 * (2. + 26. * Y2)) +
                     e2 * (135. + 4. * q2 * (-19. + 5. * Y * (-7. + 9. * Y))) +
                     3. * (45. + 2. * q2 * (-9. + Y * (-6. + 19. * Y))))) / (16. * v)
    return T, R, Th, Ph


@pytest.mark.parametrize("N", [254, 256, 258, 262142, 262144, 262146, 524290, 2103840])
def test_rates_equal_the_expressions_bit_for_bit(N):
    from emri_kludge_suite_amd import GPUAAK
    for s, p, e0, M, iota in ((0.5, 9.0, 0.2, 1e6, 0.5), (0.9, 12.0, 0.01, 2e5, 1.1), (0.0, 14.0, 0.5, 1e7, 0.3)):
        print("case rates N=%d s=%g M=%g" % (N, s, M), flush=True)
        g = GPUAAK(1.0, max(1, N // 10), N, 100.0, 15.0, True, False)
        g.set_nmax(4)
        g.gpu_gen_AAK(iota, s, p, e0, M, 10.0, 1.0, 2.0, 3.0, 1.1, 4.0, 0.7, 5.0, 1.0)
        d = g.dense_arrays()
        v, e, S, m = d["v"], d["e"], d["S"], d["M"]
        with np.errstate(all="ignore"):
            T, R, Th, Ph = _maps(v, e, np.float64(np.cos(iota)), S)
            ref = {"gimdot": (Th - R) / T / m, "Phidot": R / T / m, "alpdot": (Ph - Th) / T / m}
        good = ~(ref["Phidot"] <= 0.0)  # the guard replaces the others by the last good value
        for k in ref:
            keep = good if k == "Phidot" else slice(None)
            assert np.array_equal(d[k][keep], ref[k][keep], equal_nan=True), (k, s)
        g.close()
