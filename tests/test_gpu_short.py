"""GPU parity of the short-row transforms (single products of 2^11..2^19
points: columns of 2^D1 points by rows of 256 or 1024): products that just
fit and that just exceed half of the transform, squares, every import, and
transformed operands.  Words against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rand_limbs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", range(10, 20))
def test_nmod_depths(depth):
    import flint_amd as fa
    rng = np.random.default_rng(depth)
    n = [(1 << 61) - 1, 1000003, 0x0003F00000000001][depth % 3]
    N = 1 << depth
    for an, bn in [(N // 2, N // 2 + 1), (N // 2 + 1, 1), (N - 5, 6), (N // 3, N // 3 + 7)]:
        a = rng.integers(0, n, an, dtype=np.uint64)
        b = rng.integers(0, n, bn, dtype=np.uint64)
        zn = an + bn - 1
        print("depth %d an %d bn %d n %d" % (depth, an, bn, n), flush=True)
        want = O.nmod_poly_mul_mid(a, b, 0, zn, n)
        assert np.array_equal(fa.nmod_poly_mul_mid(a, b, 0, zn, n), want), (an, bn)
    # a square, and a window that wraps around the transform
    assert np.array_equal(fa.nmod_poly_mul_mid(a, a, 0, 2 * an - 1, n),
                          O.nmod_poly_mul_mid(a, a, 0, 2 * an - 1, n))
    a = rng.integers(0, n, N, dtype=np.uint64)
    b = rng.integers(0, n, N // 2, dtype=np.uint64)
    assert np.array_equal(fa.nmod_poly_mul_mid(a, b, N // 2 - 1, N, n),
                          O.nmod_poly_mul_mid(a, b, N // 2 - 1, N, n))


@pytest.mark.parametrize("depth", range(11, 20))
@pytest.mark.parametrize("np_,bits", [(2, 40), (4, 88), (8, 184)])
def test_mpn_depths(depth, np_, bits):
    import flint_amd as fa
    rng = np.random.default_rng(10 * depth + np_)
    limbs = (bits << depth) // 64
    an = limbs // 2 - 3
    for bn in (an, limbs - an - 3, 2, limbs // 4 + 1):
        a, b = rand_limbs(rng, an), rand_limbs(rng, bn)
        print("depth %d np %d an %d bn %d" % (depth, np_, an, bn), flush=True)
        # sums of 2 bits + 18 bits at most: every plan is exact
        assert np.array_equal(fa.mpn_mul_plan(a, b, np_, bits), O.mpn_mul(a, b)), (an, bn)


@pytest.mark.parametrize("depth", range(11, 20))
def test_fmpz_depths(depth):
    import flint_amd as fa
    rng = np.random.default_rng(depth)
    an = (1 << depth) // 2 + 1
    bn = (1 << depth) - an
    a = rng.integers(0, 2**64, 2 * an, dtype=np.uint64)
    b = rng.integers(0, 2**64, bn, dtype=np.uint64)
    got = fa.fmpz_poly_mul_mid(a, 2, b, 1, 0, an + bn - 1, 4)
    ok, want = O.fmpz_poly_mul_mid(a, 2, b, 1, 0, an + bn - 1, 4)
    assert ok and np.array_equal(got, want)


@pytest.mark.parametrize("an,bn", [(700, 600), (3000, 2500), (12000, 3000), (40000, 41000),
                                   (140000, 100000), (250000, 200000)])
def test_ops(an, bn):
    """x1 y1 - x2 y2 + x1 y1 with kept transforms of y, over the short depths
    and past them"""
    import torch
    import flint_amd as fa
    rng = np.random.default_rng(an)
    x = [rand_limbs(rng, an) for _ in range(2)]
    y = [rand_limbs(rng, bn) for _ in range(2)]
    dev = [torch.from_numpy(v.view(np.int64)).cuda() for v in x + y]
    z = torch.empty(an + bn + 1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    P = fa.Plan.mpn(an, bn, 3)
    print(an, bn, "depth", P.s.depth, flush=True)
    X = [fa.Op(P) for _ in range(4)]
    acc = fa.Op(P)
    for o, d, n in zip(X, dev, (an, an, bn, bn)):
        o.fft_mpn(d.data_ptr(), n)
    acc.mul(X[0], X[2])
    acc.addmul(X[1], X[3])
    acc.addmul(X[0], X[2])
    acc.ifft()
    acc.export_mpn(z.data_ptr(), an + bn + 1)
    fa.lib().fa_sync()
    to = lambda v: int.from_bytes(v.tobytes(), "little")
    want = 2 * to(O.mpn_mul(x[0], y[0])) + to(O.mpn_mul(x[1], y[1]))
    assert to(z.cpu().numpy()) == want
