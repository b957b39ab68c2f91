"""The law's further arithmetic of csrc/sample.hip, replayed on the CPU (fused
operations computed exactly and rounded once): e * (1/S) with one correction
and x / T by a two-part reciprocal against true division, rounding by
1.5 * 2^52 against rint, and the exp of normal results against 40 digits."""
import math
import random
import struct
from decimal import Decimal, getcontext
from fractions import Fraction

from test_law_arithmetic import K, TAB


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def test_corrected_ratio_is_true_division():
    rng = random.Random(5)
    for i in range(20000):
        S = rng.uniform(1.0, 2.0 ** rng.randint(0, 31))
        e = math.ldexp(rng.random(), -rng.choice((0, 1, 10, 100, 800, 898)))
        rS = 1.0 / S
        q = e * rS
        assert fma(fma(-q, S, e), rS, q) == e / S, (e, S)
    for S in (1.0, 2.0, 151936.0, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52, 2.0 ** 31 - 1):
        for e in (0.0, 1.0, 2.0 ** -900, 1.0 - 2.0 ** -53, 1.0 / 3):
            q = e * (1.0 / S)
            assert fma(fma(-q, S, e), 1.0 / S, q) == e / S, (e, S)
    # the remainder is subnormal: within one ulp
    for _ in range(2000):
        S, e = rng.uniform(1.0, 2.0 ** rng.randint(0, 31)), math.ldexp(rng.random(), -rng.randint(960, 1070))
        q = e * (1.0 / S)
        assert abs(fma(fma(-q, S, e), 1.0 / S, q) - e / S) <= math.ulp(e / S), (e, S)


def test_rounding_by_a_large_constant_is_rint():
    rng = random.Random(6)
    big = 1.5 * 2.0 ** 52
    values = [-0.5, -1.5, -2.5, -34430.5, 0.0, -0.0, -34441.999] + [-rng.random() * 34442 for _ in range(20000)]
    for x in values:
        assert (x + big) - big == round(x)


def test_two_part_reciprocal_is_true_division():
    rng = random.Random(7)

    def near(x, T):
        rT = 1.0 / T
        return fma(x, rT, x * (fma(-rT, T, 1.0) / T))
    for bits in range(1 << 16):                               # every finite bf16
        x = struct.unpack('<f', struct.pack('<I', bits << 16))[0]
        if math.isfinite(x):
            assert near(x, 0.8) == x / 0.8, x
    for _ in range(20000):
        x = struct.unpack('<f', struct.pack('<I', rng.getrandbits(32)))[0]
        T = 2.0 ** rng.uniform(-100, 100)
        if math.isfinite(x):
            assert near(x, T) == x / T, (x, T)


def _word(x, high_add):
    return struct.unpack('<d', struct.pack('<q', struct.unpack('<q', struct.pack('<d', x))[0] + (high_add << 32)))[0]


def exp_normal(z):
    shifted = fma(z, K['EXP_INV_L'], 1.5 * 2.0 ** 52)
    k = shifted - 1.5 * 2.0 ** 52
    n = int(k)
    r = fma(-k, K['EXP_L2'], fma(-k, K['EXP_L1'], z))
    c = fma(r, 1.0 / 720, 1.0 / 120)
    for x in (1.0 / 24, 1.0 / 6, 0.5):
        c = fma(r, c, x)
    p = fma(r * r, c, r)
    j = n & 31
    u = _word(_word(TAB[2 * j], -(j << 15)), n << 15)
    return fma(u, p + TAB[2 * j + 1] / TAB[2 * j], u)


def test_exp_of_normal_results():
    getcontext().prec = 40
    rng = random.Random(8)
    assert exp_normal(0.0) == 1.0
    worst = 0.0
    for i in range(6000):
        z = -708.0 if i == 0 else -rng.random() * (708.0, 40.0, 1.0, 1e-3)[i % 4]
        got = exp_normal(z)
        ref = Decimal(z).exp()
        worst = max(worst, float(abs(Decimal(got) - ref) / Decimal(math.ulp(float(ref)))))
    assert worst <= 0.52, worst
