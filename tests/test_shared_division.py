"""The face and grid weights' division by a shared reciprocal (csrc/divide.hpp), restated in exact
arithmetic with every step rounded once, at the ends of the range that csrc/weights.hip takes it for:
there, as inside, the quotient is the correctly rounded one, and neither it nor a step before it leaves
FP64's range."""
import math
import os
import random
import re
from fractions import Fraction

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pppm-tdbem_amd", "csrc",
                   "weights.hip")


def _limits():
    with open(SRC) as f:
        m = re.search(r"constexpr double R_MIN = (\S+), R_MAX = (\S+), Z_MAX = (\S+);", f.read())
    return float.fromhex(m[1]), float.fromhex(m[2]), float(m[3])


def _fma(a, b, c):
    """a * b + c rounded once (to nearest, subnormals kept)."""
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def _shared_div(n, d, estimate_error):
    y = float(1 / Fraction(d) * (1 + Fraction(estimate_error)))
    for _ in range(2):
        y = _fma(_fma(-d, y, 1.0), y, y)
    m = n * y
    return _fma(_fma(-d, m, n), y, m)


@pytest.mark.parametrize("r_end", ["low", "high"])
@pytest.mark.parametrize("z_end", [-1, 0, 1])
def test_quotients_at_the_ends_of_the_range(r_end, z_end):
    r_min, r_max, z_max = _limits()
    rng = random.Random(5)
    for i in range(600):
        r = (r_min if r_end == "low" else r_max) * rng.uniform(1.0, 1.001) ** (1 if r_end == "low" else -1)
        e = math.exp(z_end * z_max * rng.uniform(0.999, 1.0))
        n = e * rng.uniform(0.5, 1.0) * rng.choice((1.0, -1.0, 2.0 ** -rng.randint(1, 60)))
        for d in (4 * math.pi * r, 4 * math.pi * (r * r) * r):
            q = _shared_div(n, d, rng.uniform(-1, 1) * 2.0 ** -22)
            assert q == float(Fraction(n) / Fraction(d)), (r, n, d)
            assert 2.0 ** -1022 <= abs(q) < math.inf, (r, n, d)
