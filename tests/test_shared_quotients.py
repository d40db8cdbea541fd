"""The quotients of the FP64 sweeps: a reciprocal to an ulp, then q = a y, r = fma(-q, b, a),
fma(r, y, q).  In exact arithmetic with one rounding per operation: what lies before the last rounding
is within 2^-51 ulp of a / b, so the result is the division's but for quotients that close to the middle
between two numbers, such as some by 2 - 2^-52."""
from __future__ import annotations

import math
import random
from fractions import Fraction as Q

import pytest


def fma(a, b, c):
    return float(Q(a) * Q(b) + Q(c))


def rcp64(b, estimate):
    e = fma(-b, estimate, 1.0)
    return fma(estimate, fma(e, e, e), estimate)


def before_rounding(a, b, y):
    q = a * y
    return Q(fma(-q, b, a)) * Q(y) + Q(q)


def operands(n):
    rng = random.Random(11)
    hard = [2.0 - 2.0**-52, 1.0 + 2.0**-52, 2.0 - 2.0**-51, 1.5, 1.0, 2.0 - 2.0**-26]
    for k in range(n):
        b = hard[k] if k < len(hard) else rng.uniform(1.0, 2.0) * 2.0 ** rng.randint(-60, 60)
        # an estimate as the hardware's: 2^-24 of 1 / b off, either way
        yield b, (1.0 / b) * (1.0 + rng.uniform(-1.0, 1.0) * 2.0**-24), rng


@pytest.mark.parametrize("n", [400])
def test_quotients_round_as_divisions(n):
    off = 0
    for b, est, rng in operands(n):
        y = rcp64(b, est)
        assert abs(Q(y) * Q(b) - 1) <= Q(2) ** -52   # an ulp of 1 / b at most
        for a in [1.0, b, 3.0 * b, math.nextafter(b, 0.0)] + [rng.uniform(-2.0, 2.0) for _ in range(20)]:
            exact, got = Q(a) / Q(b), before_rounding(a, b, y)
            ulp = Q(math.ulp(a / b)) if a else Q(0)
            assert abs(got - exact) <= ulp * Q(2) ** -51
            off += float(got) != a / b
    assert off <= 2   # the divisor 2 - 2^-52 has quotients next to a middle; 9600 in all


def test_the_divisor_with_a_quotient_next_to_a_middle():
    b = 2.0 - 2.0**-52
    assert float(before_rounding(1.0, b, 0.5)) == 0.5   # y is half an ulp from 1 / b
    assert 1.0 / b == 0.5 + 2.0**-53
