"""The work that a user of this library has it do, as cases that can be timed.

Products of integers, of polynomials mod n and of integer polynomials, one call
at a time and in recorded batches, through the entry points of flint_amd.  Sizes
run from a few limbs to 2^24 limbs per operand: the ranges of the batched
workloads (flint_amd/workloads.py) and of bench.py.

Every output is a whole number of 64-bit words that the inputs determine, so
two correct implementations agree in every bit and every tolerance is "exact".
"""
import math

import numpy as np
import torch

import flint_amd as fa
from flint_amd.workloads import Rng

DEV = "cuda:0"


def listed():
    return [
        # a product of a few limbs: what one call costs before any arithmetic
        {"name": "mpn_tiny", "kind": "mpn", "an": 24, "bn": 17, "square": False},
        # an ordinary product in a computation that stays on the GPU (the
        # sizes of the smoke test): one transform of a few thousand points
        {"name": "mpn_6000x5000", "kind": "mpn", "an": 6000, "bn": 5000, "square": False},
        # a squaring, as in powering and Newton iterations
        {"name": "mpn_sqr_65536", "kind": "mpn", "an": 65536, "bn": 65536, "square": True},
        # the drop-in call on host operands (mpn_mul_default_mpn_ctx), copies
        # over PCIe included: 65,536 x 65,536 limbs
        {"name": "mpn_host_65536", "kind": "mpn_host", "an": 65536, "bn": 65536},
        # operands of odd and unequal lengths
        {"name": "mpn_ragged", "kind": "mpn", "an": 1000003, "bn": 310001, "square": False},
        # the largest single product: 2^24 x 2^24 limbs
        {"name": "mpn_2p24", "kind": "mpn", "an": 1 << 24, "bn": 1 << 24, "square": False},
        # a middle product mod n, the step of power series and division
        {"name": "nmod_mulmid", "kind": "nmod", "an": 60000, "bn": 30011, "bits": 61,
         "zl": 30010, "zh": 60000},
        # one product over Z within the eight primes
        {"name": "fmpz_9001", "kind": "fmpz", "an": 9001, "bn": 7000, "bits": 150},
        # transformed operands kept and reused: x1 y1 + x2 y2 with y1, y2 kept,
        # two forward transforms, one inverse
        {"name": "op_dot", "kind": "op", "an": 50000, "bn": 41001},
        # the batched workloads, replayed from their recorded launches
        {"name": "batch_nmod", "kind": "batch", "mix": "nmod", "count": 4096, "shapes": 3},
        {"name": "batch_fmpz", "kind": "batch", "mix": "fmpz", "count": 64, "shapes": 4},
        {"name": "batch_stream", "kind": "batch", "mix": "stream", "count": 200, "shapes": 5},
    ]


def _size(rng, lo, hi):
    """floor(2^U), U uniform in [lo, hi)"""
    return int(2 ** rng.uniform(lo, hi))


def draw(rng):
    """one more case: sizes log-uniform over the ranges above"""
    kind = rng.choice(["mpn", "mpn", "mpn", "mpn_host", "nmod", "fmpz", "op", "batch"])
    if kind == "mpn":
        an = _size(rng, 4, 24)
        square = rng.random() < 0.25
        bn = an if square else _size(rng, 4, 24)
        return {"kind": kind, "an": an, "bn": bn, "square": square}
    if kind == "mpn_host":
        return {"kind": kind, "an": _size(rng, 4, 20), "bn": _size(rng, 4, 20)}
    if kind == "nmod":
        an, bn = _size(rng, 6, 20), _size(rng, 6, 20)
        zl, zh = 0, an + bn - 1
        if rng.random() < 0.5:          # a middle product: where every term of b meets a
            zl, zh = min(an, bn) - 1, max(an, bn)
        return {"kind": kind, "an": an, "bn": bn, "bits": rng.randint(20, 63), "zl": zl, "zh": zh}
    if kind == "fmpz":
        return {"kind": kind, "an": _size(rng, 8, 14), "bn": _size(rng, 8, 14),
                "bits": _size(rng, 5, 12)}
    if kind == "op":
        return {"kind": kind, "an": _size(rng, 6, 20), "bn": _size(rng, 6, 20)}
    mix = rng.choice(["nmod", "fmpz", "stream"])
    hi = {"nmod": 12, "fmpz": 6, "stream": 7.5}[mix]
    return {"kind": kind, "mix": mix, "count": _size(rng, 2, hi), "shapes": rng.randint(6, 10**6)}


def _shapes(case):
    """(kind, an, bn, bits) of the requests of a batch, drawn as the batched
    workloads draw them"""
    r = Rng(0xF1A70000 + case["shapes"])
    out = []
    for _ in range(case["count"]):
        mix = case["mix"]
        if mix == "stream":
            u = r.double()
            mix = "mpn" if u < 0.5 else "nmod" if u < 0.8 else "fmpz"
        if mix == "mpn":
            out.append((fa.REQ_MPN, r.log_uniform(4, 22), r.log_uniform(4, 22), 0))
        elif mix == "nmod":
            out.append((fa.REQ_NMOD, r.log_uniform(6, 16), r.log_uniform(6, 16),
                        r.uniform(20, 63)))
        else:
            out.append((fa.REQ_FMPZ, r.uniform(1024, 16384), r.uniform(1024, 16384),
                        r.uniform(64, 4096)))
    return out


def _widths(kind, bits):
    """limbs per coefficient of the operands and of the output"""
    if kind != fa.REQ_FMPZ:
        return 1, 1
    return bits // 64 + 1, (2 * bits + 64) // 64 + 1


def _words(kind, an, bn, bits):
    """64-bit words of a, b and the full product"""
    w, zw = _widths(kind, bits)
    return an * w, bn * w, (an + bn if kind == fa.REQ_MPN else (an + bn - 1) * zw)


def _fill(buf, items, seed):
    """random operands at word offsets of buf: items = (offset, kind, count,
    bits, modulus)"""
    F = (fa.FillSpec * len(items))()
    r = Rng(seed)
    for f, (off, kind, count, bits, n) in zip(F, items):
        f.dst, f.count, f.kind, f.bits, f.n = buf.data_ptr() + 8 * off, count, kind, bits, n
        f.w = _widths(kind, bits)[0]
        f.key = int(fa.lib().fa_rng_next(r.s))
    torch.cuda.synchronize()            # buf comes from torch's stream
    fa.stream_fill_device(F)


def _buffer(words):
    return torch.empty(words, dtype=torch.int64, device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mpn_host":
        rng = np.random.default_rng(seed)
        return {"run": _run_host, "a": rng.integers(0, 2**64, case["an"], dtype=np.uint64),
                "b": rng.integers(0, 2**64, case["bn"], dtype=np.uint64)}
    if kind == "batch":
        return _prepare_batch(case, seed)
    an, bn = case["an"], case["bn"]
    if kind == "op":
        # two pairs of limb arrays; the plan, the ops and the transforms of
        # the kept operands are the program's
        x, y = _buffer(2 * an), _buffer(2 * bn)
        _fill(x, [(k * an, fa.REQ_MPN, an, 0, 0) for k in range(2)], seed)
        _fill(y, [(k * bn, fa.REQ_MPN, bn, 0, 0) for k in range(2)], seed + (1 << 40))
        plan = fa.Plan.mpn(an, bn, 2)
        ops = [fa.Op(plan) for _ in range(5)]
        for k in range(2):
            ops[2 + k].fft_mpn(y.data_ptr() + 8 * k * bn, bn)
        fa.lib().fa_sync()
        zn = an + bn + 1
        return {"run": _run_op, "an": an, "x": x, "y": y, "plan": plan, "ops": ops,
                "z": _buffer(zn), "zn": zn}
    bits = case.get("bits", 0)
    rk = {"mpn": fa.REQ_MPN, "nmod": fa.REQ_NMOD, "fmpz": fa.REQ_FMPZ}[kind]
    n = Rng(seed).prime(bits) if kind == "nmod" else 0
    wa, wb, wz = _words(rk, an, bn, bits)
    square = case.get("square", False)
    ab = _buffer(wa if square else wa + wb)
    items = [(0, rk, an, bits, n)] + ([] if square else [(wa, rk, bn, bits, n)])
    _fill(ab, items, seed)
    a = ab.data_ptr()
    s = {"an": an, "bn": bn, "ab": ab, "a": a, "b": a if square else a + 8 * wa}
    if kind == "mpn":
        return {**s, "run": _run_mpn, "z": _buffer(wz)}
    if kind == "nmod":
        return {**s, "run": _run_nmod, "n": n, "zl": case["zl"], "zh": case["zh"],
                "z": _buffer(case["zh"] - case["zl"])}
    w, zw = _widths(rk, bits)
    # |c| < 2^bits with both signs: the bound the program has of its operands
    return {**s, "run": _run_fmpz, "w": w, "zw": zw, "bits": bits, "z": _buffer(wz)}


def _prepare_batch(case, seed):
    shapes = _shapes(case)
    sizes = [_words(*q) for q in shapes]
    nin = sum(a + b for a, b, _ in sizes)
    ab, z = _buffer(nin), _buffer(sum(s[2] for s in sizes))
    primes = Rng(seed)
    R = (fa.Request * len(shapes))()
    items, off, zoff = [], 0, 0
    for r, (kind, an, bn, bits), (wa, wb, wz) in zip(R, shapes, sizes):
        n = primes.prime(bits) if kind == fa.REQ_NMOD else 0
        items += [(off, kind, an, bits, n), (off + wa, kind, bn, bits, n)]
        r.kind, r.an, r.bn = kind, an, bn
        r.a, r.b = ab.data_ptr() + 8 * off, ab.data_ptr() + 8 * (off + wa)
        r.z = z.data_ptr() + 8 * zoff
        off, zoff = off + wa + wb, zoff + wz
        if kind != fa.REQ_MPN:
            r.zl, r.zh = 0, an + bn - 1
        if kind == fa.REQ_NMOD:
            r.mod = fa.nmod_init(n)
        elif kind == fa.REQ_FMPZ:
            r.aw, r.zw = _widths(kind, bits)
            r.bw = r.aw
            r.abits = r.bbits = -bits
    _fill(ab, items, seed)
    batch = fa.DeviceBatch(R, graph=True, ks=True)
    if any(r.status != 1 for r in R):
        raise RuntimeError("a request of the batch was refused")
    return {"run": _run_batch, "batch": batch, "ab": ab, "z": z, "stream": fa.lib().fa_stream()}


def _run_mpn(s):
    fa.mpn_mul_device(s["z"].data_ptr(), s["a"], s["an"], s["b"], s["bn"])
    return s["z"]


def _run_host(s):
    return fa.mpn_mul(s["a"], s["b"]).view(np.int64)


def _run_nmod(s):
    fa.nmod_poly_mul_mid_device(s["z"].data_ptr(), s["zl"], s["zh"], s["a"], s["an"], s["b"],
                                s["bn"], s["n"])
    return s["z"]


def _run_fmpz(s):
    rc = fa.lib().fa_fmpz_poly_mul_mid_device(
        s["z"].data_ptr(), s["zw"], 0, s["an"] + s["bn"] - 1, s["a"], s["w"], s["an"], s["b"],
        s["w"], s["bn"], -s["bits"], -s["bits"], 1, None)
    if rc != 1:
        raise RuntimeError("fmpz product refused: %d" % rc)
    return s["z"]


def _run_op(s):
    x1, x2, y1, y2, acc = s["ops"]
    x1.fft_mpn(s["x"].data_ptr(), s["an"])
    x2.fft_mpn(s["x"].data_ptr() + 8 * s["an"], s["an"])
    acc.mul(x1, y1)
    acc.addmul(x2, y2)
    acc.ifft()
    acc.export_mpn(s["z"].data_ptr(), s["zn"])
    return s["z"]


def _run_batch(s):
    s["batch"].launch(s["stream"])
    return s["z"]


def run(state):
    return state["run"](state)


def _product_ops(points, forward=2):
    """FP64 operations of a product on `points` transform points in all (the
    points of every prime together): 4.5 per point and radix-2 level of each
    transform, 12 per point of the pointwise product"""
    depth = max(4.0, math.log2(max(points, 16)))
    return points * (4.5 * depth * (forward + 1) + 12)


def _one_work(kind, an, bn, bits, zwords):
    wa, wb, _ = _words(kind, an, bn, bits)
    # residues: 50-bit primes whose product covers twice a chunk (or
    # coefficient) and the sum over the shorter operand
    if kind == fa.REQ_MPN:
        points = 64 * (an + bn) * 2.2 / 50
    else:
        points = (an + bn) * max(1.0, (2 * bits + math.log2(min(an, bn))) / 50)
    return {"bytes": 8 * (wa + wb + zwords), "flops": _product_ops(points)}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        parts = [_one_work(*q, _words(*q)[2]) for q in _shapes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    an, bn, bits = case["an"], case["bn"], case.get("bits", 0)
    if kind == "op":
        # two operands in, two kept transforms read, one product out
        points = 64 * (an + bn) * 2.2 / 50
        return {"bytes": 8 * (2 * an + 2 * points + an + bn + 1), "flops": _product_ops(points)}
    rk = {"nmod": fa.REQ_NMOD, "fmpz": fa.REQ_FMPZ}.get(kind, fa.REQ_MPN)
    zwords = case["zh"] - case["zl"] if kind == "nmod" else _words(rk, an, bn, bits)[2]
    w = _one_work(rk, an, bn, bits, zwords)
    if case.get("square"):
        w["bytes"] -= 8 * bn
    return w


def tolerance(case):
    return "exact"


def exact(case, seed):
    """the product by Python's integers (Kronecker substitution for
    polynomials), for the sizes where that takes seconds; None elsewhere"""
    kind = case["kind"]
    if kind in ("op", "batch", "fmpz") or case["an"] + case["bn"] > 50000:
        return None
    s = prepare(case, seed)
    an, bn = case["an"], case["bn"]
    if kind == "mpn_host":
        a, b = s["a"], s["b"]
    else:
        words = s["ab"].cpu().numpy().view(np.uint64)
        a, b = words[:an], words[-bn:]
    if kind != "nmod":
        z = int.from_bytes(a.tobytes(), "little") * int.from_bytes(b.tobytes(), "little")
        return torch.from_numpy(np.frombuffer(z.to_bytes(8 * (an + bn), "little"), np.int64).copy())
    pad = np.zeros((2, max(an, bn), 3), dtype=np.uint64)
    pad[0, :an, 0], pad[1, :bn, 0] = a, b
    z = (int.from_bytes(pad[0].tobytes(), "little")
         * int.from_bytes(pad[1].tobytes(), "little")).to_bytes(24 * (an + bn), "little")
    return torch.tensor([int.from_bytes(z[24 * k:24 * k + 24], "little") % s["n"]
                         for k in range(case["zl"], case["zh"])], dtype=torch.int64)
