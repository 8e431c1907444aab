"""The adjoint's quotient by a per-type constant (div_by in diff_device.hpp): a
product with the rounded reciprocal and two corrections by the exact remainder
give the correctly rounded FP32 quotient.  The five operations are carried out
here in exact rational arithmetic, each rounded once to FP32."""
from fractions import Fraction

import numpy as np
import pytest


def _rn(x: Fraction) -> Fraction:
    """x rounded to the nearest FP32 (24 bits, ties to even; no range limit)"""
    if x == 0:
        return x
    a, e = abs(x), 0
    while a >= 1 << 24:
        a /= 2
        e += 1
    while a < 1 << 23:
        a *= 2
        e -= 1
    n = a.numerator // a.denominator
    r = a - n
    n += r > Fraction(1, 2) or (r == Fraction(1, 2) and n & 1)
    v = Fraction(n) * (Fraction(2) ** e)
    return v if x > 0 else -v


def _div_by(x, b):
    r = _rn(1 / b)
    q = _rn(x * r)
    for _ in range(2):
        q = _rn(_rn(x - b * q) * r + q)
    return q


@pytest.mark.parametrize("seed", range(4))
def test_quotient_is_correctly_rounded(seed):
    rng = np.random.default_rng(seed)
    x = np.concatenate([rng.uniform(1, 2, 800), 2.0 - 2.0 ** -23 * rng.integers(1, 9, 50),
                        1.0 + 2.0 ** -23 * rng.integers(0, 9, 50)]).astype(np.float32)
    b = np.concatenate([rng.uniform(1, 2, 800), 1.0 + 2.0 ** -23 * rng.integers(0, 9, 50),
                        2.0 - 2.0 ** -23 * rng.integers(1, 9, 50)]).astype(np.float32)
    for u, v in zip(x, rng.permutation(b)):
        u, v = Fraction(float(u)), Fraction(float(v))
        assert _div_by(u, v) == _rn(u / v), (u, v)
