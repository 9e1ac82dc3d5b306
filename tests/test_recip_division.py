"""The fused step divides by a column's areasvol and hnode_new with a reciprocal
formed once (div_by): q0 = a y, q1 = fma(fma(-b, q0, a), y, q0), q = fma(fma(-b,
q1, a), y, q1) with y = 1 / b rounded. This restates it in exact rational
arithmetic, rounding where the kernel rounds, and holds it to the correctly
rounded quotient over random operands, quotients next to a rounding boundary
and the ends of the operand ranges the kernel admits."""
import random
from fractions import Fraction as F


def _fma(a, b, c):
    return float(F(a) * F(b) + F(c))   # int/int true division rounds to nearest even


def _div_by(a, b):
    y = 1.0 / b
    q0 = a * y
    q1 = _fma(_fma(-b, q0, a), y, q0)
    return _fma(_fma(-b, q1, a), y, q1)


def _numerators(b, rng):
    """Numerators whose quotient by b lies next to the midpoint of two doubles."""
    q = rng.uniform(1.0, 2.0)
    mid = F(q) + F(1, 2 ** 53)
    a = float(mid * F(b))
    return [a, a * (1 + 2.0 ** -52), a * (1 - 2.0 ** -53), a * (1 + 2.0 ** -51)]


def test_division_by_reciprocal_is_correctly_rounded():
    rng = random.Random(11)
    for _ in range(20000):
        b = rng.uniform(1.0, 2.0) * 2.0 ** rng.randint(-30, 45)
        cases = [rng.uniform(-2.0, 2.0) * 2.0 ** rng.randint(-60, 60)] + _numerators(b, rng)
        for a in cases:
            if a != 0.0:
                assert _div_by(a, b) == a / b, (a.hex(), b.hex())
    for a in (1.1e-200, -9.9e199, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52):
        for b in (1.1e-60, 9.9e59, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52, 3.0, 6.0):
            assert _div_by(a, b) == a / b, (a.hex(), b.hex())

