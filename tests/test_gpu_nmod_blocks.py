"""Batched nmod windows at the edges of a CRT workgroup's 1024 outputs and of
its passes of 256, for one to four primes (a transform prime as modulus,
moduli of 20, 40 and 64 bits), windows inside the product, up to its end and
beyond it, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_window_edges():
    import flint_amd as fa
    rng = np.random.default_rng(0x1024)
    reqs, want = [], []
    for n in (int(fa.default_primes()[2]), 2, 1000003, (1 << 40) - 87, (1 << 64) - 59):
        an, bn = 1500, 1300
        a = (rng.integers(0, 2**63, an, dtype=np.uint64) * np.uint64(2)) % np.uint64(n)
        b = (rng.integers(0, 2**63, bn, dtype=np.uint64) * np.uint64(2) + np.uint64(1)) % np.uint64(n)
        zn = an + bn - 1
        full = O.nmod_poly_mul_mid(a, b, 0, zn, n)
        ext = np.concatenate([full, np.zeros(5000, dtype=np.uint64)])
        for cnt in (1, 255, 256, 257, 1023, 1024, 1025, 2047, 2049):
            for zl in (3, zn - cnt, zn - cnt // 2 - 1, zn - 1):
                reqs.append({"kind": "nmod", "a": a, "b": b, "n": n, "zl": zl, "zh": zl + cnt})
                want.append(ext[zl:zl + cnt])
    got = fa.batch_mul(reqs)
    for q, (st, z), w in zip(reqs, got, want):
        assert st == 1 and np.array_equal(z, w), (q["n"], q["zl"], q["zh"])
