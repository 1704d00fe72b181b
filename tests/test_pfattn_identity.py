"""The two integer identities the matrix-core prefill attention (k_pfa) is
built on, checked by brute force with Python integers (no GPU):

1. digits: sum_k x_k w_k = sum_{a+b<=13} 256^(a+b) P_ab + C sum x + C sum w - n C^2
   (mod 2^112), with S(v) the bytes of v ^ C as int8 except the top byte,
   also when some entries are the value C (all digits zero: pad positions
   and pad dims of the kernel);
2. truncated products: sum_j floor(p_j v_j / 2^48) as one FP64 sum rounding
   down for values in [-2^51, 2^51), and as three such sums for any value,
   v = v1 + 2^48 v2 (v1 = v mod 2^48), p = pa + 2^24 pb:
   sum floor(p v1 / 2^48) + sum pa v2 + 2^24 sum pb v2, every sum within
   2^51 of its start at the 4080 positions a wave has at most.

A plausible slip (the top byte offset like the others, rounding to nearest,
the split left out for large values, more positions than the bound allows)
fails one of these cases.
"""
import random
from fractions import Fraction

from test_round_down_identity import fma, rd, rn

ONE = 1 << 48
C = 0x0080808080808080
M24 = (1 << 24) - 1
START = Fraction(3 << 51)          # Q48_FSUM0
WAVE = 4080                        # positions a wave sums: 16320 / 4
EDGE = [0, 1, -1, C, -(1 << 63), (1 << 63) - 1, 1 << 48, (1 << 48) - 1, -(1 << 48),
        1 << 24, (1 << 24) - 1, 0x7F7F7F7F7F7F7F7F, 0x8080808080808080 - (1 << 64)]


def s64(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def digits(v):
    """int8 digits s_0..s_7 of v: bytes of v ^ C, top byte v's own."""
    u = (v & ((1 << 64) - 1)) ^ C
    out = []
    for i in range(8):
        b = (u >> (8 * i)) & 0xFF
        out.append(b - 256 if b >= 128 else b)
    return out


def digit_dot(xs, ws):
    dx = [digits(x) for x in xs]
    dw = [digits(w) for w in ws]
    acc = [0] * 14
    for a in range(8):
        for b in range(8):
            if a + b <= 13:
                acc[a + b] += sum(p[a] * q[b] for p, q in zip(dx, dw))
    n = len(xs)
    tot = sum(acc[d] << (8 * d) for d in range(14)) + C * sum(xs) + C * sum(ws) - n * C * C
    return tot % (1 << 112)


def fsum(ps, vs, r=rd):
    """The wave's running FP64 sum of p v, p and v as the kernel holds them, and
    the largest distance from its start."""
    acc, far = START, 0
    for p, v in zip(ps, vs):
        acc = fma(p, v, acc, r)
        far = max(far, abs(acc - START))
    return int(acc - START), far


def three_sums(ps, vs):
    """q48_f51 of v's parts, the weights' parts from p 2^-48 (pass() in k_pfa)"""
    scaled = [Fraction(p, ONE) for p in ps]
    pb = [fma(p, 1 << 24, 1 << 52) - (1 << 52) for p in scaled]
    pa = [fma(p, ONE, -b * (1 << 24)) for p, b in zip(scaled, pb)]
    assert all(a + (int(b) << 24) == p and 0 <= a < 1 << 24 for a, b, p in zip(pa, pb, ps))
    lo, hi = [v & (ONE - 1) for v in vs], [v >> 48 for v in vs]
    parts = [fsum(scaled, lo), fsum(pa, hi), fsum(pb, hi)]
    assert all(far <= 1 << 51 for _, far in parts)
    return s64(parts[0][0] + parts[1][0] + (parts[2][0] << 24))


def softmax_row(rng, n):
    """n weights in [0, ONE] that add up to at most ONE"""
    kind = rng.randrange(3)
    if kind == 0:
        return [ONE // n] * n
    cut = sorted(rng.randrange(0, ONE + 1) for _ in range(n))
    ps = [b - a for a, b in zip([0] + cut, cut)]
    return ps if kind == 1 else [p >> rng.choice([0, 0, 30]) for p in ps]


def draw(rng, edge_share=0.3):
    if rng.random() < edge_share:
        return rng.choice(EDGE)
    return rng.choice([rng.randrange(-(1 << 63), 1 << 63), rng.randrange(-(1 << 50), 1 << 50)])


def test_digit_identity_with_pads():
    rng = random.Random(3)
    for trial in range(400):
        n = rng.choice([1, 2, 5, 16, 64, 200])
        xs = [draw(rng) for _ in range(n)]
        ws = [draw(rng) for _ in range(n)]
        # pads: the value C on either side (zero digits)
        for i in range(n):
            if rng.random() < 0.1:
                xs[i] = C
        exact = sum(x * w for x, w in zip(xs, ws)) % (1 << 112)
        assert digit_dot(xs, ws) == exact, trial


def test_digit_identity_all_min():
    """every digit -128: the accumulators' largest magnitudes"""
    xs = [-(1 << 63)] * 64
    assert digit_dot(xs, xs) == sum(x * x for x in xs) % (1 << 112)


def test_value_sums_in_range():
    rng = random.Random(1)
    edge = [-(1 << 51), (1 << 51) - 1, 0, -1, 1, ONE, -ONE]
    nearest_differs = 0
    for trial in range(120):
        n = rng.choice([1, 2, 3, 17, 64, 300])
        ps = softmax_row(rng, n)
        vs = [rng.choice(edge) if trial % 3 == 0 else rng.randrange(-(1 << 51), 1 << 51)
              for _ in range(n)]
        want = sum(p * v >> 48 for p, v in zip(ps, vs))
        scaled = [Fraction(p, ONE) for p in ps]
        got, far = fsum(scaled, vs)
        assert got == want and far <= 1 << 51, trial
        nearest_differs += fsum(scaled, vs, rn)[0] != want
    assert nearest_differs > 30


def test_value_sums_of_any_value():
    rng = random.Random(4)
    whole_differs = 0
    for trial in range(120):
        n = rng.choice([1, 2, 3, 17, 64, 300])
        ps = softmax_row(rng, n)
        vs = [draw(rng) for _ in range(n)]
        want = s64(sum(p * v >> 48 for p, v in zip(ps, vs)))
        assert three_sums(ps, vs) == want, trial
        whole_differs += s64(fsum([Fraction(p, ONE) for p in ps],
                                  [rd(Fraction(v)) for v in vs])[0]) != want
    assert whole_differs > 60


def test_value_sums_at_the_longest_row():
    """Equal weights whose low 24 bits are nearly all ones, values at both ends of
    int64, as many positions as a wave sums: the low part comes to 0.96 of its
    bound, and 4400 positions would leave it."""
    p = ONE // 16305
    assert p & M24 > 0.96 * (1 << 24)
    for v in (-(1 << 63), -(1 << 63) + 1, (1 << 63) - 1):
        assert three_sums([p] * WAVE, [v] * WAVE) == s64(WAVE * (p * v >> 48))
    assert fsum([p & M24] * WAVE, [-(1 << 15)] * WAVE)[1] > 0.95 * (1 << 51)
    n = 4400
    assert fsum([p & M24] * n, [-(1 << 15)] * n)[1] > 1 << 51
