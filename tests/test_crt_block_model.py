"""CPU model of the CRT workgroup of flint_amd/csrc/fa_mpn.hip (fa_crt_fp_block,
fa_carry_resolve) and of the quotient of fa_crt_fp.h.

The workgroup cuts each coefficient into chunk-sized parts, sums the parts
that fall on a chunk, passes the excess to the next chunk, resolves the
remaining single-bit carries from generate / propagate masks, and joins the
chunks into words; the carry kernel then adds one to every block that receives
a carry.  The model replays these steps (32-bit words, 64-lane masks, blocks
of 248 chunks behind a halo of 8, segments of 16 blocks) and compares the limbs
with the integer."""
import random
from fractions import Fraction

import pytest

from oracle import oracle as O

M64 = (1 << 64) - 1


@pytest.mark.parametrize("np_", range(2, 9))
def test_quotient_by_floor(np_):
    """k = floor(sum x_i / p_i + 2^-30) in doubles is floor(S / M) or, only
    within 2^-30 M of M, one more"""
    primes = O.default_primes()[:np_]
    M = 1
    for p in primes:
        M *= p
    rng = random.Random(np_)
    edge = [0, 1, 2, M // 2, M // 2 + 1, M - 1, M - 2, M >> 29, M - (M >> 31), M - (M >> 29)]
    for c in edge + [rng.randrange(M) for _ in range(300)] + [rng.randrange(1 << 60)] * 20:
        S, qe = 0, 0.0
        for p in primes:
            x = c * pow(M // p, -1, p) % p
            if 2 * x > p:
                x -= p
            S += x * (M // p)
            qe = float(Fraction(x) * Fraction(1.0 / p) + Fraction(qe))
        k = (Fraction(qe + 2.0 ** -30)).__floor__()
        assert S - (S // M) * M == c
        r = S - k * M
        assert r == c or (r == c - M and c > M - (M >> 29)), (c, k)


def carries(G, P, c):
    """carries into 64 positions and out of the last (fa_gp_carries)"""
    X = G | P
    s = G + X + c
    return (s ^ X ^ G) & M64, s >> 64


def crt_blocks(coeffs, np_, own, zn):
    """limbs of sum_i coeffs[i] 2^(8 own i) as the kernels form them"""
    NB = (50 * np_ + 7) // 8
    OWX = (25 * np_ // 8) // 4 + 1
    bits = 8 * own
    z = [0] * zn
    nblk = (((zn + own - 1) // own) + 30) // 31
    agg = []
    for blk in range(nblk):
        rows = []
        for t in range(256):
            j = blk * 248 - 8 + t
            rows.append(coeffs[j] if 0 <= j < len(coeffs) else 0)
        S = []
        for t in range(256):
            acc, p, off = 0, 0, 0
            while off < NB:
                acc += (rows[max(t - p, 0)] >> (8 * off)) & ((1 << bits) - 1)
                p, off = p + 1, off + own
            assert p <= 7 and acc < 1 << (32 * OWX)
            S.append(acc)
        T = [(S[t] & ((1 << bits) - 1)) + (S[t - 1] >> bits if t else 0) for t in range(256)]
        G = [sum(((T[64 * w + b] >> bits) != 0) << b for b in range(64)) for w in range(4)]
        P = [sum((T[64 * w + b] == (1 << bits) - 1) << b for b in range(64)) for w in range(4)]
        for t in range(8, 256):
            assert T[t] >> bits <= 1
        G[0] &= ~0xFF
        P[0] &= ~0xFF
        c, out = 0, []
        allp = P[0] | 0xFF == M64 and all(P[w] == M64 for w in range(1, 4))
        for w in range(4):
            cin, c = carries(G[w], P[w], c)
            out += [(T[64 * w + b] + ((cin >> b) & 1)) & ((1 << bits) - 1) for b in range(64)]
        agg.append((c, int(allp)))
        data = b"".join(v.to_bytes(own, "little") for v in out[8:])
        for i in range(31 * own):
            if blk * 31 * own + i < zn:
                z[blk * 31 * own + i] = int.from_bytes(data[8 * i:8 * i + 8], "little")
    bl = 31 * own
    for blk, cin in enumerate(block_carries(agg)):
        lo, hi = blk * bl, min((blk + 1) * bl, zn)
        if cin and agg[blk][1]:
            assert z[lo:hi] == [M64] * max(hi - lo, 0)
            z[lo:hi] = [0] * max(hi - lo, 0)
        elif cin:
            for i in range(lo, hi):
                z[i] = (z[i] + 1) & M64
                if z[i]:
                    break
    return z


def byte_bits(w):
    return ((w & 0x0101010101010101) * 0x0102040810204080 & M64) >> 56


def block_carries(agg):
    """the carry into every block as fa_carry_resolve finds it: segments of 16
    blocks, the 64 blocks before one, then 2048 at a time, 32 per lane"""
    flags = [g | 2 * p for g, p in agg]
    at = lambda i: flags[i] if 0 <= i < len(flags) else 0
    out = []
    for b0 in range(0, len(agg), 16):
        c, hi = 0, b0
        if hi > 0:
            f = [at(hi - 64 + l) for l in range(64)]
            every = sum((x >> 1) << l for l, x in enumerate(f))
            _, c = carries(sum((x & 1) << l for l, x in enumerate(f)), every, 0)
            hi -= 64
            while hi > 0 and every == M64:
                G = P = 0
                for l in range(64):
                    g = p = 0
                    for k in range(4):
                        i = hi - 2048 + 32 * l + 8 * k
                        assert i % 8 == 0
                        w = sum(at(i + b) << (8 * b) for b in range(8)) if i >= 0 else 0
                        g |= byte_bits(w) << (8 * k)
                        p |= byte_bits(w >> 1) << (8 * k)
                    G |= ((g + (g | p)) >> 32) << l
                    P |= (p == 0xFFFFFFFF) << l
                _, c = carries(G, P, 0)
                every = P
                hi -= 2048
        f = [at(b0 + l) if l < 16 else 0 for l in range(64)]
        cin, _ = carries(sum((x & 1) << l for l, x in enumerate(f)),
                         sum((x >> 1) << l for l, x in enumerate(f)), c)
        out += [(cin >> l) & 1 for l in range(min(16, len(agg) - b0))]
    return out


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 80, 2111, 2112, 2113, 2129, 4300])
def test_carries_between_blocks(n):
    rng = random.Random(n)
    for k in range(12):
        agg = []
        while len(agg) < n:      # (generate, propagate): runs of ones between them
            run = int(2 ** rng.uniform(0, 12.5)) if k else n
            agg += [(rng.getrandbits(1), 0)] + [(0, 1)] * run
        agg = agg[:n]
        if k == 1:
            agg[0] = (0, 1)
        want, c = [], 0
        for g, p in agg:
            want.append(c)
            c = g | (p & c)
        assert block_carries(agg) == want


@pytest.mark.parametrize("np_,own", [(2, 3), (2, 4), (2, 6), (3, 4), (3, 9), (4, 12), (5, 15),
                                     (6, 7), (6, 16), (6, 17), (7, 21), (8, 8), (8, 25)])
def test_block_stitch(np_, own):
    rng = random.Random(100 * np_ + own)
    M = 1
    for p in O.default_primes()[:np_]:
        M *= p
    top = min(M, 1 << (16 * own + 24))
    bits = 8 * own
    for n, kind in [(1, 0), (247, 0), (248, 0), (249, 1), (700, 0), (760, 1), (760, 2), (500, 3)]:
        if kind == 0:
            c = [rng.randrange(top) for _ in range(n)]
        elif kind == 1:       # long runs of ones that a carry crosses
            c = [(1 << bits) - 1] * n
            c[rng.randrange(9)] += 1
        elif kind == 2:       # every chunk all ones, no carry
            c = [(1 << bits) - 1] * n
        else:
            c = [top - 1] * n
        zn = (bits * n + 8 * ((50 * np_ + 7) // 8)) // 64 + 1
        want = sum(v << (bits * i) for i, v in enumerate(c))
        want = [(want >> (64 * i)) & M64 for i in range(zn)]
        assert crt_blocks(c, np_, own, zn) == want, (n, kind)
        assert crt_blocks(c, np_, own, zn // 2 + 1) == want[:zn // 2 + 1], (n, kind)


def test_carries_mask():
    rng = random.Random(5)
    for _ in range(300):
        G = rng.getrandbits(64) & rng.getrandbits(64)
        P = (rng.getrandbits(64) | rng.getrandbits(64)) & ~G
        c = rng.getrandbits(1)
        got, out = carries(G, P, c)
        run = c
        for b in range(64):
            assert (got >> b) & 1 == run
            run = (G >> b) & 1 | ((P >> b) & 1 & run)
        assert out == run
