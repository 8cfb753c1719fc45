"""The CRT of integer products at every chunk width a plan may have (a
coefficient spans up to seven chunks), and the carries between its workgroups in
products with long runs of ones, where a block of ones receives a carry: words
against the closed form or the oracle, and the time against random operands of
the same lengths, single and batched."""
import math
import time

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

ONES = np.uint64(2**64 - 1)


def closed_form(n, m):
    """(B^n - 1) (B^m - 1), n >= m, B = 2^64"""
    z = np.full(n + m, ONES, dtype=np.uint64)
    z[:m] = 0
    z[0] = 1
    z[n] -= np.uint64(1)
    return z


# runs of ones that end inside a block, cross segments of 16 blocks, the 64
# before a segment, and several steps of 2048
@pytest.mark.parametrize("n,m", [(700, 700), (5001, 300), (9000, 9000), (40001, 17), (70001, 70000),
                                 (600007, 31), (1500001, 1500001), (2100003, 5)])
def test_ones(n, m):
    import flint_amd as fa
    print(n, m, fa.mpn_plan(n, m), flush=True)
    a = np.full(n, ONES, dtype=np.uint64)
    assert np.array_equal(fa.mpn_mul(a, a[:m]), closed_form(n, m))


@pytest.mark.parametrize("np_", range(2, 9))
def test_chunk_widths(np_):
    """all widths from the smallest (24 bits for two primes, 64 for eight) to the
    largest that is exact, random limbs and ones, a few blocks and part of one"""
    import flint_amd as fa
    rng = np.random.default_rng(np_)
    M = math.prod(int(p) for p in O.default_primes()[:np_])
    tried = 0
    for bits in range(24, 25 * np_ + 1, 8):
        if 9 * bits < 64 * -(-M.bit_length() // 64) + 64:
            continue
        for an, bn in ((40 * bits // 8 + 3, 23 * bits // 8), (31, 9)):
            if -(-64 * bn // bits) << 2 * bits > M:
                continue
            for a, b in ((rng.integers(0, 2**64, an, dtype=np.uint64),
                          rng.integers(0, 2**64, bn, dtype=np.uint64)),
                         (np.full(an, ONES), np.full(bn, ONES))):
                print(np_, bits, an, bn, flush=True)
                assert np.array_equal(fa.mpn_mul_plan(a, b, np_, bits), O.mpn_mul(a, b)), (bits, an)
                tried += 1
    assert tried >= 4 * (25 * np_ - 24) // 16


def runs(rng, n):
    """limbs in runs of ones, zeros and random words"""
    a = np.empty(n, dtype=np.uint64)
    i = 0
    while i < n:
        k = int(2 ** rng.uniform(0, 13))
        a[i:i + k] = [ONES, ONES, 0, rng.integers(0, 2**64, dtype=np.uint64)][rng.integers(0, 4)]
        i += k
    a[-1] |= np.uint64(1)
    return a


@pytest.mark.parametrize("an,bn", [(3000, 2), (20000, 700), (60000, 60000), (150000, 1), (200000, 9)])
def test_runs(an, bn):
    import flint_amd as fa
    rng = np.random.default_rng(an)
    pairs = []
    for k in range(4):
        a = runs(rng, an)
        b = runs(rng, bn) if k & 1 else np.full(bn, ONES, dtype=np.uint64)
        pairs.append((a, b))
    # a batch of them besides: the same kernels from a work list
    reqs = [dict(kind="mpn", a=a, b=b) for a, b in pairs]
    got = fa.batch_mul(reqs)
    for (a, b), (status, z) in zip(pairs, got):
        assert status == 1
        want = O.mpn_mul(a, b)
        assert np.array_equal(fa.mpn_mul(a, b), want)
        assert np.array_equal(z, want)


def _time(f, reps):
    import flint_amd as fa
    for _ in range(3):
        f()
    best = 1e9
    for _ in range(7):
        fa.lib().fa_sync()
        t = time.perf_counter()
        for _ in range(reps):
            f()
        fa.lib().fa_sync()
        best = min(best, (time.perf_counter() - t) / reps)
    return best


@pytest.mark.parametrize("n,count", [(1 << 16, 0), (1 << 18, 0), (1 << 22, 0), (1 << 18, 8),
                                     (1 << 20, 4)])
def test_time_on_ones(n, count):
    """(2^(64 n) - 1)^2 costs what a random square does.  Its lower half is
    blocks of ones with a carry in; turning them into zeros writes 8 n bytes
    more, under a tenth of the traffic of the product.  (One lane per block
    took 3.4, 7, 4.1 times a random square for the single ones and 2.5 and 3.6 times
    for the batches.)"""
    import torch
    import flint_amd as fa
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    k = max(count, 1)
    rand = torch.randint(-2**63, 2**63 - 1, (k * n,), generator=g, device="cuda")
    z = torch.empty(2 * k * n, dtype=torch.int64, device="cuda")
    t = []
    for a in (rand, torch.full_like(rand, -1)):
        torch.cuda.synchronize()
        if count:
            R = (fa.Request * k)()
            for i, r in enumerate(R):
                r.kind, r.an, r.bn = fa.REQ_MPN, n, n
                r.a = r.b = a.data_ptr() + 8 * n * i
                r.z = z.data_ptr() + 16 * n * i
            B = fa.DeviceBatch(R)
            s = fa.lib().fa_stream()
            t.append(_time(lambda: B.launch(s), 5))
            B.close()
        else:
            t.append(_time(lambda: fa.mpn_mul_device(z.data_ptr(), a.data_ptr(), n, a.data_ptr(), n),
                           10))
        print("%d x %d limbs: %.1f us" % (k, n, 1e6 * t[-1]), flush=True)
    assert t[1] < 1.5 * t[0]
