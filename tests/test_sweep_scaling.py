"""Rewrites of the reference-rounding sweep that change no bit, on the CPU.

  * division by 3, 6, 12, 18 and 24 as RN(x h + RN(x l)), h = RN(1/c),
    l = RN(1/c - h), in exact rational arithmetic against the correctly rounded
    quotient: random operands, multiples of the divisor, all-ones
    significands, operands next to the quotients' rounding boundaries, zeros, the
    smallest operands of the bound that the code states and those below it;
  * the last step of the reciprocal, in exact rational arithmetic;
  * the WENO5 side on doubled arguments with four times eps: exactly twice the
    side on the arguments themselves, weights bit for bit (NumPy doubles),
    from 1e-140 to 1e45; a wrong eps fails.
"""
import re
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest

MATH = Path(__file__).resolve().parents[1] / "how-mhd-kokkos_amd" / "csrc" / "mhd_math.hpp"


def _rn(f):
    return f.numerator / f.denominator  # int / int is correctly rounded


def _two_step(x, c):
    h = 1.0 / c
    lo = _rn((1 - Fraction(c) * Fraction(h)) / c)
    return lo, _rn(Fraction(x) * Fraction(h) + Fraction(x * lo))


@pytest.mark.parametrize("c", [3, 6, 12, 18, 24])
def test_division_by_constant(c):
    rng = np.random.default_rng(c)
    xs = list(rng.standard_normal(4000) * 10.0 ** rng.integers(-280, 280, 4000))
    for _ in range(2000):
        m = int(rng.integers(1 << 52, 1 << 53))
        e = int(rng.integers(-200, 200))
        xs += [float(m) * 2.0 ** e, float(m // c * c) * 2.0 ** e, float((1 << 53) - 1 - int(rng.integers(0, 9))) * 2.0 ** e]
        # next to c times a midpoint of two doubles
        xs += [_rn(Fraction(2 * m + 1, 2) * c + k) for k in (-1, 0, 1)]
    for x in xs:
        assert _two_step(x, c)[1] == _rn(Fraction(x) / c), x.hex()
    lo, _ = _two_step(1.0, c)
    assert lo > 0.0
    h = 1.0 / c
    for x in (0.0, -0.0):  # the sum of products keeps the sign of a zero
        assert np.signbit(x * h + x * lo) == np.signbit(x / c)


# divisor -> its least operand of the stated bound that the margin gives (1/18 and
# 1/6 ulp against a rounding error of 2^-1075)
_LEAST = {3: 3.0 * 2.0 ** -1020, 6: 6.0 * 2.0 ** -1020, 12: 12.0 * 2.0 ** -1020, 18: 18.0 * 2.0 ** -1018,
          24: 24.0 * 2.0 ** -1020}


@pytest.mark.parametrize("c", [3, 6, 12, 18, 24])
def test_division_by_constant_smallest_operands(c):
    """Every binade from the bound that the code states up to 2^-1000, and the four
    above the divisor's own: the correctly rounded quotient.  Below, for any
    operand, one of the two doubles next to the quotient."""
    text = MATH.read_text().split("x / c for a compile-time constant")[1]
    bound = 2.0 ** -int(re.search(r"\|x\| >= 2\^-(\d+)", text).group(1))
    assert bound >= _LEAST[c]
    rng = np.random.default_rng(100 + c)

    def binade(lo, n):
        return np.concatenate([lo * (1.0 + rng.random(n)), [lo, np.nextafter(lo, np.inf)]])

    lows = [2.0 ** -e for e in range(1000, -int(np.log2(bound)) + 1)] + [_LEAST[c] * 2.0 ** k for k in range(4)]
    for lo in lows:
        for x in binade(lo, 2000):
            x = float(x)
            assert _two_step(x, c)[1] == _rn(Fraction(x) / c), x.hex()
    for e in range(1014, 1075):
        for x in 2.0 ** -e * (1.0 + rng.random(50)):
            got, exact = _two_step(float(x), c)[1], Fraction(float(x)) / c
            assert Fraction(np.nextafter(got, -np.inf)) < exact < Fraction(np.nextafter(got, np.inf))


def test_reciprocal_step():
    """The last step of recip_rn from either double next to 1/b: the correctly
    rounded reciprocal, but for the all-ones significand from the double below."""
    rng = np.random.default_rng(3)
    ms = [int(m) for m in rng.integers(1 << 52, 1 << 53, 20000)]
    ms += [(1 << 52) + k for k in range(1, 200)] + [(1 << 53) - k for k in range(1, 200)]
    for m in ms:
        b = m * 2.0 ** -52
        exact = 1 / Fraction(b)
        want = _rn(exact)
        below = want if Fraction(want) < exact else float(np.nextafter(want, 0.0))
        for r in (below, float(np.nextafter(below, 1.0))):
            d = 1 - Fraction(b) * Fraction(r)
            assert Fraction(_rn(d)) == d  # the remainder is a double
            got = _rn(Fraction(r) + Fraction(r) * d)
            assert (got == want) != (m == (1 << 53) - 1 and r == below), b.hex()


def _side(a, b, c, d, eps):
    is0 = 13.0 * (a - b) * (a - b) + 3.0 * (a - 3.0 * b) * (a - 3.0 * b)
    is1 = 13.0 * (b - c) * (b - c) + 3.0 * (b + c) * (b + c)
    is2 = 13.0 * (c - d) * (c - d) + 3.0 * (3.0 * c - d) * (3.0 * c - d)
    t = [(eps + s) * (eps + s) for s in (is0, is1, is2)]
    al = [1.0 / t[0], 6.0 / t[1], 3.0 / t[2]]
    s = al[0] + al[1] + al[2]
    w0, w2 = al[0] / s, al[2] / s
    return w0, w2, w0 * (a - 2.0 * b + c) / 3.0 + (w2 - 0.5) * (b - 2.0 * c + d) / 6.0


def test_doubled_weno_side():
    rng = np.random.default_rng(1)
    n = 200000
    v = rng.standard_normal((4, n)) * 10.0 ** rng.uniform(-140, 45, n)
    v[:, ::3] = v[0, ::3] * (1.0 + 1e-6 * rng.standard_normal((4, v[:, ::3].shape[1])))  # smooth
    v[rng.integers(0, 4, n // 7), np.arange(n // 7)] = 0.0
    v[:, -1] = 0.0
    w0, w2, phi = _side(*v, 1.0e-10)
    x0, x2, twice = _side(*(2.0 * v), 4.0 * 1.0e-10)
    for a, b in ((w0, x0), (w2, x2), (2.0 * phi, twice)):
        assert np.array_equal(a.view(np.int64), b.view(np.int64))
    assert not np.array_equal(_side(*(2.0 * v), 1.0e-10)[2], twice)
