"""Products of one small transform around the line between interleaved and
separate operands (256 points), and at both ends of the former's range:
integer, nmod and fmpz imports, against exact integers and the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.golden.make_fixtures import poly_ks
from tests.helpers import rand_limbs, to_int
from tests.test_gpu_ks import dec, draw, enc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("an,bn", [(1, 1), (2, 1), (24, 17), (150, 120), (300, 1), (330, 300),
                                   (400, 390), (700, 40)])
def test_mpn(an, bn):
    import flint_amd as fa
    rng = np.random.default_rng(an * 31 + bn)
    a, b = rand_limbs(rng, an), rand_limbs(rng, bn)
    for x, y in ((a, b), (b, a), (a, a)):
        assert to_int(fa.mpn_mul(x, y)) == to_int(x) * to_int(y)


@pytest.mark.parametrize("an,bn", [(1, 1), (2, 1), (3, 5), (100, 29), (128, 128), (128, 129),
                                   (129, 129), (200, 57), (250, 270)])
def test_poly(an, bn):
    import flint_amd as fa
    rng = np.random.default_rng(an * 37 + bn)
    n = (1 << 63) - 25
    a = rng.integers(0, n, an, dtype=np.uint64)
    b = rng.integers(0, n, bn, dtype=np.uint64)
    zn = an + bn - 1
    assert np.array_equal(fa.nmod_poly_mul_mid(a, b, 0, zn, n),
                          O.nmod_poly_mul_mid(a, b, 0, zn, n))
    u, v = draw(rng, an, 100, "mixed"), draw(rng, bn, 60, "mixed")
    z = fa.fmpz_poly_mul_mid(enc(u, 2), 2, enc(v, 1), 1, 0, zn, 3)
    assert dec(z, 3) == poly_ks(u, v, signed=True)
