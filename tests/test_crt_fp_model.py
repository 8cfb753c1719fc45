"""CPU model of the radix-2^24 FP64 CRT of flint_amd/csrc/fa_crt_fp.h
(fa_crt_fp_value).

The GPU kernel forms sum_i x_i (M/p_i) - k M with exact FP64 FMAs on 24-bit
digits, x_i in [-p/2, p/2], k = floor(sum_i x_i / p_i + 2^-30).  This model
replays the same steps on Python integers and asserts, at every FMA and carry
step, that the value is an integer below 2^53 (so the double operation is
exact), that the products of the two halves of x_i stay below 2^48 and 2^49, and
that the sign correction is taken exactly where k is one more than the quotient.
The recombined coefficient is checked against the residues' defining integer for
every prime count 2..8, at random, near 0, M/2 and M, and within 2^-30 M of M,
where the correction is taken; and the two centred parts (the signed exports).
"""
import random
from fractions import Fraction

import pytest

from oracle import oracle as O

B = 1 << 24


def _exact(v):
    assert v.denominator == 1 and abs(v) < 2 ** 53, v
    return float(v)


def _digits(x, nd):
    return [float((x >> (24 * d)) & 0xFFFFFF) for d in range(nd)]


def crt_fp_model(xs, primes):
    np_ = len(primes)
    M = 1
    for p in primes:
        M *= p
    ND = (50 * np_ + 23) // 24
    NDC = (50 * (np_ - 1) + 23) // 24
    cof = [_digits(M // p, 16) for p in primes]
    Md, h = _digits(M, 18), _digits(M // 2, 18)
    assert all(c == 0 for row in cof for c in row[NDC:]) and all(c == 0 for c in Md[ND:])
    rp = [1.0 / p for p in primes]
    col = [0.0] * ND

    def carry():
        c = 0.0
        for m in range(ND):
            v = _exact(Fraction(col[m]) + Fraction(c))
            c = float((Fraction(v) / B).__floor__())
            col[m] = _exact(Fraction(v) - Fraction(c) * B)
        return c

    qe = 0.0
    for i, x in enumerate(xs):
        if i == 6:
            top = carry()
            col[ND - 1] = _exact(Fraction(col[ND - 1]) + Fraction(top) * B)
        x = float(x)
        assert 2 * abs(x) <= primes[i]
        qe = float(Fraction(x) * Fraction(rp[i]) + Fraction(qe))   # one rounding (fma)
        v = float(int(x) >> 24)
        u = _exact(Fraction(x) - Fraction(v) * B)
        for d in range(NDC):
            assert u * cof[i][d] < 2 ** 48 and abs(v * cof[i][d]) < 2 ** 49
            col[d] = _exact(Fraction(u) * Fraction(cof[i][d]) + Fraction(col[d]))
            col[d + 1] = _exact(Fraction(v) * Fraction(cof[i][d]) + Fraction(col[d + 1]))
    k = float(Fraction(qe + 2.0 ** -30).__floor__())
    for m in range(ND):
        col[m] = _exact(Fraction(col[m]) - Fraction(k) * Fraction(Md[m]))
    S = sum(x * (M // p) for x, p in zip(xs, primes))
    top = carry()
    assert top == (-1 if k > S // M else 0) and k - S // M in (0, 1)
    if top < 0:
        for m in range(ND):
            col[m] = _exact(Fraction(col[m]) + Fraction(Md[m]))
        carry()
    value = lambda c: sum(int(c[m]) << (24 * m) for m in range(ND))
    # MODE 1 and 2: the positive and the negated negative part of the centred value
    gt = next((col[m] > h[m] for m in range(ND - 1, -1, -1) if col[m] != h[m]), False)
    pos = 0 if gt else value(col)
    c, neg = value(col), 0
    if gt:
        col = [Md[m] - col[m] for m in range(ND)]
        carry()
        neg = value(col)
    return c, pos, neg, top < 0


@pytest.mark.parametrize("np_", range(2, 9))
def test_crt_fp_model_exact(np_):
    primes = [int(p) for p in O.default_primes()[:np_]]
    M = 1
    for p in primes:
        M *= p
    cofinv = [pow(M // p % p, -1, p) for p in primes]
    rs = random.Random(np_)
    cases = [0, 1, M - 1, M // 2, M // 2 - 1, M // 2 + 1, M // 3]
    cases += [rs.randrange(M) for _ in range(60)]
    cases += [rs.randrange(2 ** 40) for _ in range(10)]
    cases += [M - 1 - rs.randrange(2 ** 40) for _ in range(10)]
    cases += [M - (M >> 32) - rs.randrange(M >> 40) for _ in range(5)]    # corrected
    cases += [M - (M >> 28) - rs.randrange(M >> 40) for _ in range(5)]    # not
    corrected = 0
    for c in cases:
        xs = [c * cofinv[i] % primes[i] for i in range(np_)]
        xs = [x - p if 2 * x > p else x for x, p in zip(xs, primes)]
        got, pos, neg, fix = crt_fp_model(xs, primes)
        assert got == c
        assert (pos, neg) == ((0, M - c) if c > M // 2 else (c, 0))
        assert fix == (c > M - (M >> 30)) or M - (M >> 29) < c < M - (M >> 31)
        corrected += fix
    assert corrected >= 16
