"""CPU model of the nmod CRT of flint_amd/csrc/fa_poly.hip (fa_crt_nmod_value).

The kernel finds the mixed-radix digits t_k of the coefficient c in [0, M) with
FP64 mulmods (h = a b, q = rint(h / p), r = fma(-q, p, h) + fma(a, b, -h)) and
the reductions that their bounds need, then c mod n by Horner's rule with
128-bit products.  The double operations are replayed exactly (FMA through
rationals, rint half-even), with every mulmod's operands below 4 p^2, every
running value within the bounds stated at the kernel, every digit in [0, p), the
high word below n at every 128-bit reduction, and the result equal to c mod n:
for every prime count 1..8 at every offset into the eight default primes, stored
residues anywhere in [-8p, 8p], c at its extremes and of any length, and moduli
n from 1 to 2^64 - 59."""
import random
from fractions import Fraction

import pytest

from oracle import oracle as O


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def _pm1n(a, p, pinv):
    return _fma(-float(round(a * pinv)), p, a)


def _consts(primes):
    M = 1
    for p in primes:
        M *= p
    gcm = [(M // p) % p for p in primes]
    ginv, gpm = [], []
    for k, pk in enumerate(primes):
        pre, row = 1 % pk, []
        for j in range(k):
            row.append(primes[j] % pk)
            pre = pre * (primes[j] % pk) % pk
        gpm.append(row)
        ginv.append(pow(pre, pk - 2, pk))
    return M, gcm, ginv, gpm


def _mulmod(a, b, p, pinv):
    assert abs(int(a) * int(b)) < 4 * int(p) ** 2
    h = a * b
    r = _fma(-float(round(h * pinv)), p, h) + _fma(a, b, -h)
    assert r == int(r) and (int(r) - int(a) * int(b)) % int(p) == 0
    return r


def digits(xs, primes):
    _, gcm, ginv, gpm = _consts(primes)
    t = []
    for k, pk in enumerate(primes):
        p, pinv = float(pk), 1.0 / pk
        r = _mulmod(_pm1n(float(xs[k]), p, pinv), float(gcm[k]), p, pinv)
        assert abs(r) <= 0.75 * p
        y = r
        if k:
            u = t[k - 1]
            for i in range(k - 2, -1, -1):
                u = _mulmod(u, float(gpm[k][i]), p, pinv) + t[i]
                assert abs(u) <= 3.5 * p and u == int(u)
            if k > 2:
                u = _pm1n(u, p, pinv)
            y = _pm1n(_mulmod(r - u, float(ginv[k]), p, pinv), p, pinv)
        t.append(y + p if y < 0 else y)
        assert 0 <= t[k] < p
    return [int(x) for x in t]


@pytest.mark.parametrize("np_", range(1, 9))
def test_digits_exact(np_):
    P = [int(p) for p in O.default_primes()]
    rnd = random.Random(100 + np_)
    for off in range(0, 9 - np_):
        primes = P[off:off + np_]
        M = 1
        for p in primes:
            M *= p
        for trial in range(60):
            c = (rnd.randrange(M), M - 1 - rnd.randrange(1000), rnd.randrange(1000),
                 M // 2 + rnd.randrange(-5, 5),
                 rnd.randrange(1 << rnd.randint(1, M.bit_length() - 1)))[trial % 5]
            xs = [c * pow((M // p) % p, p - 2, p) % p + p * rnd.randrange(-8, 8) for p in primes]
            t = digits(xs, primes)
            n = rnd.choice([1, 2, 3, (1 << 64) - 59, (1 << 63) + 29, rnd.randrange(2, 1 << 64),
                            rnd.randrange(2, 1 << 20)])
            v = t[-1] if np_ > 1 else t[-1] % n
            for k in range(np_ - 2, -1, -1):
                w = v * (primes[k] % n) + t[k]
                assert (w >> 64) < n
                v = w % n
            assert v == c % n
