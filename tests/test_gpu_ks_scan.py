"""The flag scan and the packing of the signed-slot Kronecker route where they
can go wrong: lengths around a wave, 1024 and a round of 4096 coefficients,
runs of zero coefficients that carry a borrow across waves and rounds, the top
coefficient far below the end, all-zero operands, slots just below, at and
above 64 bits, coefficients of the largest magnitude.  The expected words are
those of the exact product, by substitution into Python integers.  And the time
on an operand that is zero above its first coefficient."""
import time

import numpy as np
import pytest

from tests.golden.make_fixtures import poly_ks
from tests.test_gpu_ks import dec, draw, enc

pytestmark = pytest.mark.gpu

#        an,  bits a, bits b, pattern
CASES = [(63, 200, 90, "dense"), (64, 130, 64, "lowzero"), (65, 29, 29, "dense"),
         (1023, 30, 30, "sparse"), (1024, 31, 30, "dense"), (1025, 64, 63, "sparse"),
         (4095, 100, 20, "run"), (4096, 128, 127, "run"), (4097, 190, 64, "run"),
         (8200, 65, 40, "run"), (4500, 90, 64, "lead"), (5000, 640, 70, "extreme"),
         (3000, 80, 80, "zero")]


def fill(rng, n, bits, pattern):
    v = draw(rng, n, bits, "mixed")
    if pattern == "sparse":
        v = [x if rng.integers(0, 9) == 0 else 0 for x in v]
    elif pattern == "lowzero":      # low limbs zero
        v = [(x >> 128) << 128 for x in v]
    elif pattern == "run":          # one borrow through a run of zeros
        v = [-5] + [0] * (n - 2) + [7]
    elif pattern == "lead":         # the top coefficient (negative) far below the end
        v = v[:n // 9] + [-3] + [0] * (n - n // 9 - 1)
    elif pattern == "extreme":
        v = [(1 << bits) - 1 if x >= 0 else 1 - (1 << bits) for x in v]
    elif pattern == "zero":
        v = [0] * n
    return v


@pytest.mark.parametrize("an,abits,bbits,pattern", CASES)
def test_flags_and_packing(an, abits, bbits, pattern):
    import flint_amd as fa
    rng = np.random.default_rng(an + abits)
    a = fill(rng, an, abits, pattern)
    b = draw(rng, 9, bbits, "mixed")
    b[3] = b[4] = 0
    aw, bw, zw = abits // 64 + 1, bbits // 64 + 1, (abits + bbits + 6) // 64 + 1
    zn = an + 8
    want = poly_ks(a, b, signed=True) if any(a) else [0] * zn
    for x, xw, y, yw in ((a, aw, b, bw), (b, bw, a, aw)):
        z = fa.fmpz_poly_mul_ks(enc(x, xw), xw, enc(y, yw), yw, 0, zn + 1, zw)
        assert dec(z, zw) == want + [0]
    lo = zn - zn // 3
    z = fa.fmpz_poly_mul_ks(enc(a, aw), aw, enc(b, bw), bw, lo, zn, zw)
    assert dec(z, zw) == want[lo:]


def test_time_of_leading_zeros():
    """the flags of an operand whose coefficients above the first are zero: each
    zero coefficient's limbs are read once, so the product takes what one with
    only top limbs set takes (1.28 times that with two walks)"""
    import torch
    import flint_amd as fa
    n, bits = 9000, 3900
    w, zw = bits // 64 + 1, (2 * bits + 64) // 64 + 1
    z = torch.empty((2 * n - 1) * zw, dtype=torch.int64, device="cuda")
    t = []
    for top in (True, False):
        a = torch.zeros((n, w), dtype=torch.int64, device="cuda")
        if top:
            a[:, -1] = 1
        else:
            a[0, 0] = 5
        torch.cuda.synchronize()
        best = 1e9
        for _ in range(12):
            s = time.perf_counter()
            for _ in range(3):
                assert fa.lib().fa_fmpz_poly_mul_mid_device(
                    z.data_ptr(), zw, 0, 2 * n - 1, a.data_ptr(), w, n, a.data_ptr(), w, n, -bits,
                    -bits, 1, None) == 1
            fa.lib().fa_sync()
            best = min(best, (time.perf_counter() - s) / 3)
        t.append(best)
    print("us", [round(1e6 * x) for x in t], flush=True)
    assert t[1] < 1.15 * t[0]
