"""The quotient of a march step of SSR (multiply by the refined reciprocal, two fused
corrections, the range test on the divisor alone), step by step in exact arithmetic
rounded to binary32: correctly rounded for every numerator of 2^-110 and more, and below
2^-50 where it is not."""
import random
from fractions import Fraction

import numpy as np


def _round(x):
    """A Fraction to the nearest binary32 (ties to even, subnormals kept)."""
    if x == 0:
        return np.float32(0)
    m = abs(x)
    e = m.numerator.bit_length() - m.denominator.bit_length()
    e = max(e - 1 if Fraction(2) ** e > m else e, -126)
    ulp = Fraction(2) ** (e - 23)
    n = round(m / ulp)                     # Fraction rounds ties to even
    return np.float32(float((n if x > 0 else -n) * ulp))


def _fma(a, b, c):
    return _round(Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c)))


def test_march_quotient():
    rng = random.Random(1)
    wrong = checked = 0
    for _ in range(12000):
        ea, ed = rng.randint(-149, -20), rng.randint(-60, 60)
        if ea - ed > 0:
            continue
        a = np.float32(rng.uniform(1, 2) * 2.0 ** ea) if ea > -127 else \
            np.float32(rng.randint(1, 2 ** min(23, ea + 150)) * 2.0 ** -149)
        d = np.float32(rng.choice([-1, 1]) * rng.uniform(1, 2) * 2.0 ** ed)
        r0 = _round(1 / Fraction(float(d)))
        if rng.random() < 0.5:             # v_rcp_f32 is within one ulp
            r0 = np.nextafter(r0, np.float32(rng.choice([-1e30, 1e30])), dtype=np.float32)
        r = _fma(_fma(-d, r0, 1.0), r0, r0)
        q = _round(Fraction(float(a)) * Fraction(float(r)))
        q = _fma(_fma(-d, q, a), r, q)
        q = _fma(_fma(-d, q, a), r, q)
        want = _round(Fraction(float(a)) / Fraction(float(d)))
        checked += 1
        if q != want:
            wrong += 1
            assert a < 2.0 ** -110 and abs(want) < 2.0 ** -50 and abs(q) < 2.0 ** -50
            assert abs(float(q) - float(want)) <= max(2.0 ** -149, 2.0 ** -23 * abs(float(want)))
    assert checked > 5000 and wrong > 0
