"""The flag scan and the packing of the signed-slot Kronecker route where they
can go wrong: lengths around a wave, 1024 and a round of 4096 coefficients,
runs of zero coefficients that carry a borrow across waves and rounds, the top
coefficient far below the end, all-zero operands, slots just below, at and
above 64 bits, coefficients of the largest magnitude.  The expected words are
those of the exact product, by substitution into Python integers."""
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
