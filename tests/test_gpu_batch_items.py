"""Work items of a batch's transforms, which name blocks of adjacent column
tiles and rows: every column length, whole and truncated to row counts that end
inside a block, against the oracle; and what making a batch takes."""
import time

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rand_limbs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d1", [1, 2, 3, 4, 5, 7, 9])
def test_blocks_and_truncated_rows(d1):
    """products of 2^(12 + d1) points that end 1, 3 and 2^(d1 - 1) - 1 rows past the
    half, and that fill the transform"""
    import flint_amd as fa
    rng = np.random.default_rng(d1)
    half = 1 << (d1 - 1)
    reqs = []
    for rows in sorted({min(half + k, 2 * half) for k in (1, 3, half - 1, half)}):
        if rows == half:
            continue
        limbs = 88 * 4096 * rows // 64 - 3
        an = limbs // 2 + 1
        for trunc in (fa.TRUNC_ON, fa.TRUNC_OFF):
            reqs.append(dict(kind="mpn", a=rand_limbs(rng, an), b=rand_limbs(rng, limbs - an),
                             np=4, bits=88, trunc=trunc))
    got = fa.batch_mul(reqs)
    for q, (status, z) in zip(reqs, got):
        assert status == 1
        assert np.array_equal(z, O.mpn_mul(q["a"], q["b"])), (len(q["a"]), q["trunc"])


def test_time_of_making_a_batch():
    """making a batch of 1024 products of 2^13 points, of which 1000 coefficients
    are asked for, against one of 1024 products of 32 points: 1.6 times (2.5 times
    with one item per tile)"""
    import torch
    import flint_amd as fa
    N, n = 1024, (1 << 61) - 1
    a = torch.randint(0, n, (1 << 12,), device="cuda")
    z = torch.empty(1000 * N, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    t = []
    for an in (16, 1 << 12):
        R = (fa.Request * N)()
        for i, r in enumerate(R):
            r.kind, r.an, r.bn, r.mod = fa.REQ_NMOD, an, an, fa.nmod_init(n)
            r.a = r.b = a.data_ptr()
            r.z = z.data_ptr() + 8000 * i
            r.zl, r.zh = 0, min(1000, 2 * an - 1)
        best = 1e9
        for _ in range(25):
            s = time.perf_counter()
            B = fa.DeviceBatch(R)
            best = min(best, time.perf_counter() - s)
            B.close()
        t.append(best)
    print("us", [round(1e6 * x) for x in t], flush=True)
    assert t[1] < 2.1 * t[0]
