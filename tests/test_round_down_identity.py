"""The FP64 forms that round toward minus infinity (csrc/q48_device.hpp:
q48_round_down, q48_exp_small, q48_recip, q48_divisor_of / q48_div_by,
q48_inv_sqrt), restated with every operation rounded down from its exact
rational value and checked against integer arithmetic (no GPU).  Each check
also shows that rounding to nearest, the mode the switch replaces, or a
dropped compare gives wrong values here.
"""
import math
import random
from fractions import Fraction

ONE = 1 << 48
M64 = (1 << 64) - 1


def rd(x):
    """The largest double at or below the rational x (|x| in the normal range)."""
    x = Fraction(x)
    if x == 0:
        return x
    e = abs(x.numerator).bit_length() - x.denominator.bit_length() - 54
    ulp = Fraction(2) ** e
    while abs(x) / ulp >= 1 << 53:
        ulp *= 2
    return math.floor(x / ulp) * ulp


def rn(x):
    return Fraction(float(Fraction(x)))


def fma(a, b, c, r=rd):
    return r(Fraction(a) * Fraction(b) + Fraction(c))


H52 = Fraction(1 << 52)


def exp_squares(m, n, r=rd):
    h, out = H52 + ONE + (m >> 14), []
    for _ in range(n):
        y = fma(h, Fraction(1, 1 << 24), -(1 << 28), r)
        h = fma(y, y, H52, r)
        out.append(int(h - H52))
    return out


def newton2(d, rel):
    dd = rd(d)
    y = rn(Fraction(1) / dd * (1 + Fraction(rel)))
    for _ in range(2):
        y = fma(y, fma(-dd, y, 1), y)
    return y


def quotient(num_low, y, scale, e, d, compare=True):
    h = fma(e, y * scale, H52 - Fraction(1, 2))
    q0 = (math.floor(h - H52)) & M64     # 2^52 - 1/2 gives -1, as its word does
    rem = (num_low - q0 * d) & M64
    up = compare and rem >= d
    if rem - (d if up else 0) >= d:
        return None
    return (q0 + up) & M64


def inv_sqrt_steps(xn, y, r=rd):
    M = Fraction(3 << 51)
    xs = Fraction(xn, 1 << 48)
    cx = M - M * xs
    assert rd(cx) == cx
    tq = ((3 << 48) + M) / (1 << 49)
    for _ in range(7):
        t1 = fma(y, Fraction(y) / ONE, M, r)
        t2 = fma(t1, xs, cx, r)
        fs = fma(t2, Fraction(-1, 1 << 49), tq, r)
        y = fma(y, fs, M, r) - M
        if not 1 <= y < 1 << 49:
            return None
    return int(y)


def inv_sqrt_ref(xn, y):
    for _ in range(7):
        f = (3 << 48) - (xn * ((y * y) >> 48) >> 48)
        y = y * f >> 49
        if y <= 0:
            return 1
    return y


def test_squarings():
    rng = random.Random(1)
    ms = [0, 1, 10 * ONE, 10 * ONE - 1, ONE, 5 * ONE]
    ms += [rng.randrange(0, 10 * ONE + 1) >> rng.choice([0, 0, 20, 40]) for _ in range(800)]
    nearest_differs = 0
    for m in ms:
        ref, want = ONE + (m >> 14), []
        for _ in range(12):
            ref = ref * ref >> 48
            want.append(ref)
        assert exp_squares(m, 12) == want and want[-1] < 1 << 52, m
        nearest_differs += exp_squares(m, 12, rn) != want
    assert nearest_differs > len(ms) // 2


def test_reciprocals():
    rng = random.Random(2)
    rs = [ONE, ONE + 1, (1 << 63) - 1, 1 << 62, int(22026.47 * ONE)]
    rs += [rng.randrange(ONE, 1 << 63) for _ in range(1500)]
    rs += [min(max((1 << 96) // q + dd, ONE), (1 << 63) - 1)
           for q in (rng.randrange(1 << 33, 1 << 48) for _ in range(500)) for dd in (-1, 0, 1)]
    short = 0
    for r in rs:
        y = newton2(r, (rng.random() - 0.5) * 2.0 ** -19)
        assert quotient(0, y, Fraction(2) ** 96, 1, r) == (1 << 96) // r, r
        short += quotient(0, y, Fraction(2) ** 96, 1, r, compare=False) != (1 << 96) // r
    assert short > 100


def test_prepared_divisors():
    rng = random.Random(3)
    cases = [(0, 1), (1, 1), ((1 << 52) - 1, (1 << 52) - 1), (ONE, ONE), (0, (1 << 62) - 1),
             ((1 << 52) - 1, (1 << 62) - 1)]
    for _ in range(1500):
        d = max(1, rng.randrange(1, 1 << 62) >> rng.randrange(0, 62))
        cases.append((rng.randrange(0, min(d, (1 << 52) - 1) + 1), d))
    for _ in range(700):   # softmax rows, and next to exact quotients
        d = rng.randrange(ONE, 4097 * ONE)
        e = rng.randrange(0, ONE + 1) * d >> 48
        cases += [(min(max(e + dd, 0), (1 << 52) - 1), d) for dd in (-1, 0, 1)]
        cases.append((rng.randrange(0, ONE + 1), d))
    for e, d in cases:
        y48 = rd(newton2(d, (rng.random() - 0.5) * 2.0 ** -19) * ONE)
        assert quotient(e << 48, y48, 1, e, d) == (e << 48) // d, (e, d)


def test_inv_sqrt_steps():
    rng = random.Random(4)
    xs = [ONE, ONE + 1, 2 * ONE - 1, 2 * ONE, 4 * ONE - 1]
    xs += [ONE + (rng.randrange(3 * ONE) >> rng.choice([0, 0, 20, 45])) for _ in range(400)]
    nearest_differs = 0
    for xn in xs:
        y = ((3 << 48) - xn) >> 1 if xn < 2 * ONE else ((3 << 48) - (xn >> 2)) >> 2
        want = inv_sqrt_ref(xn, y)
        assert inv_sqrt_steps(xn, y) == want, xn
        nearest_differs += inv_sqrt_steps(xn, y, rn) != want
    assert nearest_differs > 10
