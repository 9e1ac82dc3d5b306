"""The fused step divides by 3 and 6 with the constant's reciprocal in two parts:
fma(a, zh, a zl), zh = RN(1/c), zl = RN(1/c - zh), for numerators of at least
1e-280 (smaller ones are divided). This restates it in exact rational
arithmetic, rounding where the kernel rounds, and holds it to the correctly
rounded quotient over random numerators, quotients next to a rounding boundary
and the ends of the range."""
import random
from fractions import Fraction as F

import pytest

PARTS = {3: (float.fromhex("0x1.5555555555555p-2"), float.fromhex("0x1.5555555555555p-56")),
         6: (float.fromhex("0x1.5555555555555p-3"), float.fromhex("0x1.5555555555555p-57"))}


def _fma(a, b, c):
    return float(F(a) * F(b) + F(c))   # a Fraction's conversion rounds to nearest even


@pytest.mark.parametrize("c", [3, 6])
def test_two_part_reciprocal_is_correctly_rounded(c):
    zh, zl = PARTS[c]
    assert zh == 1.0 / c and zl == float(F(1, c) - F(zh))
    rng = random.Random(c)
    cases = [1e-280, 1.7e308, 2.0 ** -900, 1.0, 3.0, 6.0, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52]
    for _ in range(20000):
        a = rng.uniform(-2.0, 2.0) * 2.0 ** rng.randint(-900, 900)
        q = rng.uniform(1.0, 2.0)
        mid = float((F(q) + F(1, 2 ** 53)) * c)   # a numerator whose quotient is next to a midpoint
        cases += [a, mid, mid * (1 + 2.0 ** -52), mid * (1 - 2.0 ** -53)]
    for a in cases:
        assert _fma(a, zh, a * zl) == a / c, a.hex()
