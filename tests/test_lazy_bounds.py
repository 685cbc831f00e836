"""The FP64 kernels' lazy arithmetic (csrc/modarith.hpp) at its bounds: every value is an integer of at most 8 p
<= 2^53.  The products and reductions are evaluated here in IEEE doubles (the fused multiply-add through exact
rationals) on operands at the ends of their ranges, and the forward transform's schedule is driven with
the largest values that each stage can give; csrc/modarith.hpp and csrc/ksfused.hip assert the same
recurrence at compile time."""

import random
import re
from fractions import Fraction

import pytest

from holmes_amd import build as hb

MODULI = [(1 << 50) - 27 * (1 << 17) + 1, (1 << 50) - 1, (1 << 49) + 1, (1 << 40) + 15, 6 * (1 << 17) + 1]
CENTERED = 0.5 + 2.0**-10


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))  # correctly rounded


def mulv(a, b, p, pinv):
    h = a * b
    q = float(round(h * pinv))
    low = fma(a, b, -h)
    assert Fraction(low) == Fraction(a) * Fraction(b) - Fraction(h)
    return _exact_sum(fma(-q, p, h), -Fraction(q) * Fraction(p) + Fraction(h), low)


def mulc(a, w, wp, p):
    q = float(round(a * wp))
    h = a * w
    low = fma(a, w, -h)
    return _exact_sum(fma(-q, p, h), -Fraction(q) * Fraction(p) + Fraction(h), low)


def _exact_sum(x, exact, low):
    assert Fraction(x) == exact, "the multiply-add has to be exact"
    assert Fraction(x + low) == exact + Fraction(low), "the final sum has to be exact"
    return x + low


def reduce(x, p, pinv):
    q = float(round(x * pinv))
    r = fma(-q, p, x)
    assert Fraction(r) == Fraction(x) - Fraction(q) * Fraction(p)
    return r


def canon(x, p, pinv):
    r = reduce(x, p, pinv)
    return r + p if r < 0.0 else r


def _operands(rng, top, p, n=40):
    """Integers of at most `top`, the ends of the range among them."""
    ends = [0, 1, -1, top, -top, top - 1, 1 - top]
    return [float(v) for v in ends + [rng.randint(-top, top) for _ in range(n)] + [rng.randint(top - p // 2, top)
                                                                                   for _ in range(n)]]


@pytest.mark.parametrize("p", MODULI)
def test_products_and_reductions_hold_to_eight_p(p):
    rng = random.Random(p)
    fp, pinv = float(p), 1.0 / float(p)
    top = min(8 * p - 1, 1 << 53)
    ws = [0, 1, p - 1, p // 2, p // 2 + 1] + [rng.randrange(p) for _ in range(8)]
    for a in _operands(rng, top, p):
        A = abs(a) / p
        c = canon(a, fp, pinv)
        assert 0 <= c < p and (int(c) - int(a)) % p == 0
        assert abs(reduce(a, fp, pinv)) <= p / 2 + 2
        for w in ws:
            r = mulv(a, float(w), fp, pinv)
            assert (int(r) - int(a) * w) % p == 0 and abs(r) <= (0.5 + 0.375 * A) * p + 1
            r = mulc(a, float(w), float(w) / fp, fp)
            assert (int(r) - int(a) * w) % p == 0 and abs(r) <= (0.5 + 0.25 * A) * p + 1


def test_forward_schedule_at_its_largest_values():
    """The values of a stage come from disjoint inputs, so the largest sum operand meets the largest
    product: driven with those, all sixteen stages stay exact below 8 p."""
    src = (hb.CSRC / "modarith.hpp").read_text()
    body = re.search(r"constexpr bool fwd_reduces\(int l\) \{ return (.*?); \}", src)[1]
    reduces = {int(v) for v in re.findall(r"l == (\d+)", body)}
    p = MODULI[0]
    fp, pinv = float(p), 1.0 / float(p)
    rng = random.Random(7)
    for start in (p - 1, p // 2 + 512):  # canonical words, centered words
        bound = start / p
        largest = float(start)
        for stage in range(16):
            m = 0.0
            for _ in range(60):
                v = largest - rng.randrange(1 << 20)
                m = max(m, abs(mulv(v, float(p - 1 - rng.randrange(1 << 20)), fp, pinv)),
                        abs(mulv(v, float(rng.randrange(p)), fp, pinv)))
            u = float(p // 2 + 512) if stage in reduces else largest
            bound = (CENTERED if stage in reduces else bound) + 0.5 + 0.375 * bound
            largest = u + m
            assert Fraction(largest) == Fraction(u) + Fraction(m)
            assert largest <= bound * p < 8 * p, stage
        assert bound < 5.61


@pytest.mark.parametrize("dropped", [3, 6, 9, 11, 14])
def test_each_reduction_is_needed(dropped):
    """One reduction fewer takes a bound past 8 p: the schedule has no slack to lose."""
    a = 1.0
    peak = 0.0
    for stage in range(16):
        a = (0.5 if stage in {3, 6, 9, 11, 14} - {dropped} else a) + 0.5 + 0.375 * a
        peak = max(peak, a)
    assert peak > 8.0
