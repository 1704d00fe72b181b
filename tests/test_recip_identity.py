"""The quotients of csrc/q48_device.hpp around their FP64 estimates (q48_recip,
q48_exp_neg, q48_divisor_of / q48_div_by), restated with every FP64 operation
rounded down as on the device, checked against integer arithmetic (no GPU):

1. fp_safe_exp(-u) for 0 <= u as q48_exp_neg makes it: 12 squarings on
   doubles, two on integers, and floor(2^96 / r) without q48_recip's fallback
   to the general division;
2. two Newton steps are needed and enough, whatever first approximation within
   2^-20 the hardware gives: one step leaves remainders that one compare does
   not settle, which q48_recip and q48_div_by would send to the general
   division and q48_exp_neg would get wrong;
3. the divisor's range: at d = 2^62 - 1 and e = 2^52 - 1 the estimate still
   settles, and every divisor of a softmax row does.

The forms' values over their whole ranges are in test_round_down_identity.py.
"""
import math
import random
from fractions import Fraction

from test_round_down_identity import M64, ONE, exp_squares, fma, quotient, rd, rn

H52 = Fraction(1 << 52)


def newton(d, rel, steps):
    dd = rd(d)
    y = rn(Fraction(1) / dd * (1 + Fraction(rel)))
    for _ in range(steps):
        y = fma(y, fma(-dd, y, 1), y)
    return y


def remainder(num_low, y, scale, e, d):
    """The estimate's remainder word: below 2 d where the compare settles it"""
    q0 = math.floor(fma(e, y * scale, H52 - Fraction(1, 2)) - H52) & M64
    return (num_low - q0 * d) & M64


def fp_exp(m):
    """fp_exp(-m) of the reference (fp_math.h:724-732), m >= 0"""
    r = ONE + (m >> 14)
    for _ in range(14):
        r = r * r >> 48
    return (1 << 96) // r


def exp_neg(u, rel, steps=2):
    lim = 10 * ONE
    m = min(u, lim)
    r = exp_squares(m, 12)[-1]
    for _ in range(2):
        r = r * r >> 48
    q = quotient_no_fallback(r, newton(r, rel, steps))
    return q if u <= lim else 0


def quotient_no_fallback(r, y):
    q0 = math.floor(fma(1, y * Fraction(2) ** 96, H52 - Fraction(1, 2)) - H52) & M64
    rem = -q0 * r & M64
    return (q0 + (1 if rem >= r else 0)) & M64


def rel20(rng):
    return (rng.random() - 0.5) * 2.0 ** -19


def test_exp_neg():
    rng = random.Random(1)
    us = [0, 1, 1 << 14, 10 * ONE - 1, 10 * ONE, 10 * ONE + 1, ONE, (1 << 63) - 1]
    us += [rng.randrange(0, 10 * ONE + 1) >> rng.choice([0, 0, 8, 30]) for _ in range(1500)]
    for u in us:
        want = fp_exp(u) if u <= 10 * ONE else 0
        assert exp_neg(u, rel20(rng)) == want, u


def test_newton_steps():
    rng = random.Random(2)
    one_short = 0
    for _ in range(800):
        r = rng.randrange(ONE, 1 << 63)
        assert remainder(0, newton(r, rel20(rng), 2), Fraction(2) ** 96, 1, r) < 2 * r
        one_short += quotient(0, newton(r, 2.0 ** -20, 1), Fraction(2) ** 96, 1, r) is None
    assert one_short > 0


def test_divisor_range():
    rng = random.Random(3)
    cases = [((1 << 52) - 1, (1 << 62) - 1), ((1 << 52) - 1, (1 << 52) - 1), (0, (1 << 62) - 1)]
    for _ in range(800):    # softmax rows: e <= ONE <= sum <= 16320 ONE
        cases.append((rng.randrange(0, ONE + 1), rng.randrange(ONE, 16320 * ONE)))
    for e, d in cases:
        y48 = rd(newton(d, rel20(rng), 2) * ONE)
        assert remainder(e << 48, y48, 1, e, d) < 2 * d, (e, d)
        assert quotient(e << 48, y48, 1, e, d) == (e << 48) // d, (e, d)
