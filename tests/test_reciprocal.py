"""The kernels' reciprocal of an axis, 1 / (2n + 1), is the IEEE quotient.

Kernels take the hardware's approximate reciprocal r (within 1 ulp) and one
Newton step, fma(fma(-d, r, 1), r, r).  Exact rational arithmetic with one
rounding per operation shows that the step gives the nearest float of 1/d for
every d = 2n + 1 a level can have (n < 65536) from any r within 2 ulp.
"""
from fractions import Fraction

import numpy as np


def _round(x: Fraction) -> float:
    """Nearest float32 of x > 0 (ties to even; none occur), by rounding its 24-bit mantissa."""
    e = 0
    while x * Fraction(2) ** e < 1 << 23:
        e += 8
    while x * Fraction(2) ** e >= 1 << 24:
        e -= 1
    return float(Fraction(round(x * Fraction(2) ** e)) / Fraction(2) ** e)


def test_newton_step_gives_the_ieee_quotient():
    for n in list(range(1, 600)) + list(range(600, 65536, 37)) + [32767, 65534, 65535]:
        d = 2 * n + 1
        q = np.float32(1.0) / np.float32(d)
        bits = q.view(np.uint32)
        for ulp in (-2, -1, 0, 1, 2):
            r = (bits + np.uint32(ulp % (1 << 32))).view(np.float32) if ulp >= 0 else (bits - np.uint32(-ulp)).view(np.float32)
            fr = Fraction(float(r))
            e = 1 - d * fr  # exact in float32: a difference of near-equal numbers of few bits, rounded below
            e32 = Fraction(0) if e == 0 else (Fraction(_round(e)) if e > 0 else -Fraction(_round(-e)))
            assert _round(e32 * fr + fr) == float(q), (n, ulp)
