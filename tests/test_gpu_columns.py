"""GPU parity of the column passes where their import and first stage branch:
operands of more and of less than half the transform, every piece count of a
byte-aligned chunk, operands that end inside a 32-byte window or are shorter
than one, u64 coefficients on both sides of 2^50, and signed coefficients of
one to four limbs at their extremes.  Words against the oracle."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rand_limbs

pytestmark = pytest.mark.gpu

# (np, bits): 1, 2, 3, 4 and 5 pieces of 48 bits
PLANS = [(2, 40), (3, 64), (4, 88), (6, 136), (8, 184), (8, 192)]


@pytest.mark.parametrize("np_,bits", PLANS)
@pytest.mark.parametrize("depth", [13, 14, 16, 17, 18])
def test_mpn_import(depth, np_, bits):
    """one operand past half the transform (no zero half), the other of one
    limb to half of it; lengths that end at every offset of a window"""
    import flint_amd as fa
    rng = np.random.default_rng(1000 * depth + bits)
    limbs = (bits << depth) // 64            # limbs of a full transform
    for k, bn in enumerate([1, 3, 4, 5, limbs // 3]):
        an = limbs - bn - (k * 7) % 11 - 1
        a, b = rand_limbs(rng, an), rand_limbs(rng, bn)
        if k == 2:
            a[:] = b[:] = np.uint64(0xFFFFFFFFFFFFFFFF)
        print("depth %d np %d bits %d an %d bn %d" % (depth, np_, bits, an, bn), flush=True)
        # exact while the primes' product holds the sum over the shorter operand
        M = math.prod(int(p) for p in O.default_primes()[:np_])
        if min(-(-64 * n // bits) for n in (an, bn)) << 2 * bits > M:
            with pytest.raises(fa.FlintAmdError, match="error -4: .*not exact"):
                fa.mpn_mul_plan(a, b, np_, bits)
            continue
        assert np.array_equal(fa.mpn_mul_plan(a, b, np_, bits), O.mpn_mul(a, b)), (an, bn)


@pytest.mark.parametrize("n", [998244353, (1 << 50) - 27, (1 << 63) - 25])
@pytest.mark.parametrize("an,bn", [(5000, 3), (4096, 4096), (8191, 1), (60000, 1234),
                                   (70000, 60001)])
def test_nmod_import(an, bn, n):
    import flint_amd as fa
    fa.lib().fa_set_direct_fft(0)
    try:
        rng = np.random.default_rng(an + bn)
        a = rng.integers(0, n, an, dtype=np.uint64)
        b = rng.integers(0, n, bn, dtype=np.uint64)
        a[-1] = b[-1] = n - 1
        print(an, bn, n, flush=True)
        got = fa.nmod_poly_mul_mid(a, b, 0, an + bn - 1, n)
    finally:
        fa.lib().fa_set_direct_fft(1)
    assert np.array_equal(got, O.nmod_poly_mul_mid(a, b, 0, an + bn - 1, n))


@pytest.mark.parametrize("w", [1, 2, 3, 4])
def test_fmpz_import(w):
    """coefficients of w limbs: all bits random, and the extremes
    -2^(64 w - 20), 2^(64 w - 20) - 1 and -1"""
    import flint_amd as fa
    rng = np.random.default_rng(w)
    an, bn = 9001, 2
    aw, bw, zw = w, 1, w + 2
    a = rng.integers(0, 2**64, (an, aw), dtype=np.uint64)
    a[:, -1] = (a[:, -1].astype(np.int64) >> 20).astype(np.uint64)
    lo = np.zeros(aw, dtype=np.uint64)
    lo[-1] = np.int64(-(1 << 44)).astype(np.uint64)
    a[0], a[1], a[2], a[-1] = lo, ~lo, ~np.zeros(aw, dtype=np.uint64), lo
    b = rng.integers(0, 1 << 30, (bn, bw), dtype=np.uint64)
    b[1] = ~np.uint64(0)                   # -1
    got = fa.fmpz_poly_mul_mid(a.ravel(), aw, b.ravel(), bw, 0, an + bn - 1, zw)
    ok, want = O.fmpz_poly_mul_mid(a.ravel(), aw, b.ravel(), bw, 0, an + bn - 1, zw)
    assert ok and got is not None and np.array_equal(got, want)
