"""The constant divisions of the equilibrium, written as a multiply and a fused multiply-add
(over_cs2, over_cs2x2 and over_cs4x2 in madpac_amd/csrc/lbm_cell.h), against the correctly rounded
quotient, in exact rational arithmetic: random significands, and the quotients nearest to a rounding
boundary, found by solving 2^k X = t (mod C) for small t."""
from fractions import Fraction

import numpy as np
import pytest


def rounded(v: Fraction) -> Fraction:
    """v rounded to the nearest double, ties to even (normal range)."""
    if v == 0:
        return v
    a = abs(v)
    e = a.numerator.bit_length() - a.denominator.bit_length()
    while Fraction(2) ** e > a:
        e -= 1
    ulp = Fraction(2) ** (e - 52)
    return (1 if v > 0 else -1) * round(a / ulp) * ulp


@pytest.mark.parametrize("divisor, z, zl", [
    (1.0 / 3.0, 3.0, float.fromhex("0x1.8p-53")),
    (2.0 * (1.0 / 3.0), 1.5, float.fromhex("0x1.8p-54")),
    (2.0 * (1.0 / 3.0) * (1.0 / 3.0), 4.5, float.fromhex("0x1.2p-52")),
])
def test_division_by_constants_is_correctly_rounded(divisor, z, zl):
    c, z, zl = Fraction(divisor), Fraction(z), Fraction(zl)
    rng = np.random.default_rng(3)
    xs = [int(v) | 1 << 52 for v in rng.integers(0, 1 << 52, 4000)] + [1 << 52, (1 << 53) - 1]
    C = c.numerator
    while C % 2 == 0:
        C //= 2
    for t in list(range(-8, 0)) + list(range(1, 9)):
        for k in range(60):
            x0 = t * pow(2, -k, C) % C
            xs += [x for x in range(x0, 1 << 53, C) if x >= 1 << 52][:4]
    assert len(xs) > 4500
    for x in xs:
        for v in (Fraction(x), -Fraction(x)):
            assert rounded(z * v + rounded(zl * v)) == rounded(v / c)


def test_division_of_the_coupling_force_is_correctly_rounded():
    # over_cs4: (c.u)^2 / ((1.0/3.0)*(1.0/3.0))
    test_division_by_constants_is_correctly_rounded((1.0 / 3.0) * (1.0 / 3.0), 9.0, float.fromhex("0x1.2p-51"))
