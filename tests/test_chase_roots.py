"""The short chains for a root and its reciprocal in the chase's reflector give the
IEEE-rounded square root and quotient (a CPU model of the iteration, with exact fused
multiply-adds, over estimates as coarse as 2^-20)."""
import math
import random
from fractions import Fraction


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def _sqrt_and_recip(x, est):
    g, h = x * est, 0.5 * est
    r = _fma(-h, g, 0.5)
    g, h = _fma(g, r, g), _fma(h, r, h)
    for _ in range(2):
        g = _fma(_fma(-g, g, x), h, g)
    v = 2.0 * h
    for _ in range(2):
        v = _fma(_fma(-g, v, 1.0), v, v)
    return g, v


def test_root_and_reciprocal_are_rounded_as_ieee():
    rng = random.Random(1)
    for t in range(4000):
        x = rng.uniform(1.0, 4.0) if t % 2 else math.ldexp(rng.uniform(1.0, 2.0), rng.randint(-699, 699))
        if t % 5 == 0:  # squares and their neighbours: roots at and near representable values
            x = float(rng.randint(1, 1 << 26)) ** 2
            x = math.nextafter(x, math.inf) if hasattr(math, "nextafter") and t % 10 == 0 else x
        est = (1.0 / math.sqrt(x)) * (1.0 + rng.uniform(-1, 1) * 2.0**-20)
        root, inv = _sqrt_and_recip(x, est)
        assert root == math.sqrt(x), x
        assert inv == 1.0 / root, x
