"""Batched nmod windows at the edges of a CRT workgroup's 256 or 1024 outputs
(batches below a million outputs, and from there on) and of its passes of 256,
for one to four primes (a transform prime as modulus, moduli of 20, 40 and 64
bits), windows inside the product, up to its end and beyond it, against the
oracle; and what the kernel takes for a small batch."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("more", [0, 1 << 20])
def test_window_edges(more):
    import flint_amd as fa
    rng = np.random.default_rng(0x1024)
    reqs, want = [], []
    if more:
        x = np.arange(1, more // 2 + 2, dtype=np.uint64)
        reqs.append({"kind": "nmod", "a": x, "b": x, "n": 1000003, "zl": 0, "zh": more + 1})
        want.append(O.nmod_poly_mul_mid(x, x, 0, more + 1, 1000003))
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


def test_time_of_small_batch():
    """the CRT kernel of a batch of one product of 999 coefficients takes what
    that of the single call takes, 6.3 us between events (with four outputs per
    thread it took 7.1)"""
    import torch
    import flint_amd as fa
    n, an = (1 << 61) - 1, 500
    a = torch.randint(0, n, (an,), device="cuda")
    z = torch.empty(2 * an, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    R = (fa.Request * 1)()
    r = R[0]
    r.kind, r.an, r.bn, r.a, r.b, r.z = fa.REQ_NMOD, an, an, a.data_ptr(), a.data_ptr(), z.data_ptr()
    r.zl, r.zh, r.mod = 0, 2 * an - 1, fa.nmod_init(n)
    B = fa.DeviceBatch(R, graph=False)
    s = fa.lib().fa_stream()

    def both():
        B.launch(s)
        fa.nmod_poly_mul_mid_device(z.data_ptr(), 0, 2 * an - 1, a.data_ptr(), an, a.data_ptr(), an,
                                    n, s)
    for _ in range(20):
        both()
    fa.lib().fa_sync()
    ratio = []
    for _ in range(7):
        fa.prof_reset()
        fa.prof_enable(True)
        for _ in range(100):
            both()
        fa.prof_enable(False)
        p = fa.prof_read()
        ratio.append(p["fa_kb_crt_nmod"][0] / p["fa_k_crt_nmod"][0])
    B.close()
    print(ratio, flush=True)
    assert min(ratio) < 1.07
