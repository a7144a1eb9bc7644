"""Performance cases of the multiply and of what a program builds on it.

Each case is one call (or one short sequence of calls) as a program that keeps
its numbers on the GPU makes it, through the library's public entry points:
products from the schoolbook range to 2^24 words, squares, multiply-adds in
batches, a captured batch, host-array products, the fft.h sequence, division
and radix conversion. Operand words are uniform, either in [0, 1e9) (the
benchmark's operands) or over all 32 bits (what binary splitting and Newton
steps produce), made on the GPU from the seed.

Kinds and their ranges:
  mul     one product, al x bl words, 16 .. 2^24 each (balanced and uneven)
  sqr     one square, 50 .. 2^23 words
  host    one product of host arrays (the drop-in use: words copied in and
          out over the link), 500 .. 2^21 words
  level   one bcg_muladd_batch_dev call: `count` independent P0 Q1 + P1 of
          nearly equal lengths around `words` (a binary-splitting level)
  replay  a captured batch of `count` products with log-uniform lengths in
          [16, top], replayed (bcg_batch_run)
  chain   int_to_fft of two operands, two forward transforms, pointwise
          product, inverse transform, fft_to_int (the fft.h sequence of the
          reference's own multiply), points = 2^k or 3 2^k
  div     device bigfloat quotient a / b at precision p (Newton reciprocal)
  radix   base-1e9 digits of a binary fraction of `words` words
"""
import ctypes
import math
import random

import numpy as np
import torch

import bluecrunch_amd as bc


def listed():
    return [
        # the smallest calls: one schoolbook product, latency only
        {"name": "mul_24x19", "kind": "mul", "al": 24, "bl": 19, "full": True},
        # a few thousand digits: a Newton step's or exp's ordinary small product
        {"name": "mul_1000x777", "kind": "mul", "al": 1000, "bl": 777, "full": True},
        # a million digits, the plain single multiply of the benchmark set
        {"name": "mul_2p17", "kind": "mul", "al": 1 << 17, "bl": 1 << 17, "full": False},
        # ragged operands of unlike lengths (division and radix steps)
        {"name": "mul_300007x41003", "kind": "mul", "al": 300007, "bl": 41003, "full": True},
        # the largest single product of the benchmark set
        {"name": "mul_2p24", "kind": "mul", "al": 1 << 24, "bl": 1 << 24, "full": False},
        # an odd-sized large square (powering, Newton iterations)
        {"name": "sqr_3000017", "kind": "sqr", "al": 3000017, "full": True},
        # the drop-in call of a C program: host words in, host words out
        {"name": "host_1000003", "kind": "host", "al": 1000003, "bl": 1000003, "full": True},
        # one level of a binary-splitting tree: equal-length multiply-adds
        {"name": "level_256x3001", "kind": "level", "count": 256, "words": 3001},
        # many small uneven products, captured once and replayed
        {"name": "replay_4096", "kind": "replay", "count": 4096, "top": 16384},
        # the transform entry points in the order the reference's multiply calls them
        {"name": "chain_2p20", "kind": "chain", "points": 1 << 20, "bits": 12},
        # a quotient to about a million digits
        {"name": "div_100003", "kind": "div", "p": 100003},
        # ten million digits out of a binary fraction
        {"name": "radix_1038145", "kind": "radix", "words": 1038145},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mul", "mul", "mul", "sqr", "sqr", "host", "level", "replay", "chain", "div", "radix"])
    full = rng.random() < 0.6
    if kind == "mul":
        al = _log(rng, 16, 1 << 24)
        bl = al if rng.random() < 0.4 else _log(rng, max(16, al // 64), al)
        return {"kind": "mul", "al": al, "bl": bl, "full": full}
    if kind == "sqr":
        return {"kind": "sqr", "al": _log(rng, 50, 1 << 23), "full": full}
    if kind == "host":
        al = _log(rng, 500, 1 << 21)
        return {"kind": "host", "al": al, "bl": _log(rng, max(100, al // 16), al), "full": full}
    if kind == "level":
        words = _log(rng, 100, 200000)
        return {"kind": "level", "count": _log(rng, 2, max(2, min(1024, 1600000 // words))), "words": words}
    if kind == "replay":
        return {"kind": "replay", "count": _log(rng, 64, 4096), "top": _log(rng, 256, 16384)}
    if kind == "chain":
        n = 1 << rng.randint(10, 22)
        return {"kind": "chain", "points": n if rng.random() < 0.6 else 3 * n // 4, "bits": rng.randint(8, 12)}
    if kind == "div":
        return {"kind": "div", "p": _log(rng, 200, 200000)}
    return {"kind": "radix", "words": _log(rng, 500, 1 << 20)}


# ------------------------------------------------------------------ operands

def _words(gen, n, full=True):
    """n device words, uniform in [0, 2^32) or [0, 1e9), as int32 bits."""
    hi = (1 << 32) if full else 10 ** 9
    w = torch.randint(0, hi, (n,), generator=gen, device="cuda", dtype=torch.int64)
    w[-1] = torch.clamp(w[-1], min=1)
    return w.to(torch.int32)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & 0x7FFFFFFF)
    return g


def _offsets(n):
    return np.concatenate([[0], np.cumsum(n)[:-1]]).astype(np.uint64)


def _sizes(x):
    return np.ascontiguousarray(x, dtype=np.uint64)


def _level_lengths(case):
    """Lengths of P0, Q1 and P1 for each product of a tree level: the nodes of
    one level differ by a few words."""
    r = random.Random(case["count"] * 1000003 + case["words"])
    w = case["words"]
    spread = max(1, w // 50)
    pick = lambda: np.array([w - r.randrange(spread) for _ in range(case["count"])], dtype=np.int64)  # noqa: E731
    return pick(), pick(), pick()


def _replay_lengths(case):
    """Two log-uniform operand lengths in [16, top] for each product."""
    r = random.Random(case["count"] * 7919 + case["top"])
    one = lambda: [_log(r, 16, case["top"]) for _ in range(case["count"])]  # noqa: E731
    return np.array(one(), dtype=np.int64), np.array(one(), dtype=np.int64)


class _Words:
    """A torch tensor seen as the device words of a library call."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    s = {"kind": kind, "case": case}
    if kind in ("mul", "sqr"):
        al = case["al"]
        bl = case["bl"] if kind == "mul" else al
        s["a"] = _words(gen, al, case["full"])
        s["b"] = _words(gen, bl, case["full"]) if kind == "mul" else s["a"]
        s["c"] = torch.empty(al + bl, dtype=torch.int32, device="cuda")
    elif kind == "host":
        s["a"] = _words(gen, case["al"], case["full"]).cpu().numpy().view(np.uint32)
        s["b"] = _words(gen, case["bl"], case["full"]).cpu().numpy().view(np.uint32)
    elif kind == "level":
        pl, ql, dl = _level_lengths(case)
        cl = pl + ql + 1
        s["a"] = _words(gen, int(pl.sum()))
        s["b"] = _words(gen, int(ql.sum()))
        s["d"] = _words(gen, int(dl.sum()))
        s["c"] = torch.empty(int(cl.sum()), dtype=torch.int32, device="cuda")
        s["args"] = [_sizes(x) for x in (_offsets(cl), cl, _offsets(pl), pl, _offsets(ql), ql, _offsets(dl), dl)]
    elif kind == "replay":
        al, bl = _replay_lengths(case)
        cl = al + bl
        s["a"] = _words(gen, int(al.sum()), False)
        s["b"] = _words(gen, int(bl.sum()), False)
        s["c"] = torch.empty(int(cl.sum()), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()  # the library runs on a stream of its own
        s["batch"] = bc.Batch(_Words(s["c"]), _Words(s["a"]), _Words(s["b"]), _offsets(cl), cl, _offsets(al), al,
                              _offsets(bl), bl)
    elif kind == "chain":
        n = case["points"]
        # each operand fills half of the points, as a product's operands do
        w = n * case["bits"] // 64
        s["a"] = _words(gen, w)
        s["b"] = _words(gen, w)
        s["za"] = torch.empty(2 * n, dtype=torch.float64, device="cuda")
        s["zb"] = torch.empty(2 * n, dtype=torch.float64, device="cuda")
        s["c"] = torch.empty(2 * w, dtype=torch.int32, device="cuda")
    elif kind == "div":
        p = case["p"]
        a = _words(gen, p).cpu().numpy().view(np.uint32).copy()
        b = _words(gen, p).cpu().numpy().view(np.uint32).copy()
        a[-1] |= 0x80000000  # a / b in (1, 4): the quotient's length does not hang on the seed
        b[-1] = (b[-1] | 0x40000000) & 0x7FFFFFFF
        s["a"] = bc.DeviceBigfloat((a, -p, 1))
        s["b"] = bc.DeviceBigfloat((b, -p, 1))
        s["t"] = bc.DeviceBigfloat()
    elif kind == "radix":
        n = case["words"]
        s["f"] = _words(gen, n)
        s["groups"] = max(1, int((n - 3) / 0.9343253125117121))
        s["d"] = torch.empty(s["groups"], dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()  # the library runs on a stream of its own
    return s


def run(s):
    kind = s["kind"]
    L = bc.lib()
    if kind in ("mul", "sqr"):
        a, b, c = s["a"], s["b"], s["c"]
        bc.mul_dev(c.data_ptr(), c.numel(), a.data_ptr(), a.numel(), b.data_ptr(), b.numel())
        return c
    if kind == "host":
        return bc.mul(s["a"], s["b"])[0]
    if kind == "level":
        ptrs = [x.ctypes.data_as(ctypes.POINTER(ctypes.c_size_t)) for x in s["args"]]
        worst = ctypes.c_double()
        bc.check(L.bcg_muladd_batch_dev(s["c"].data_ptr(), s["a"].data_ptr(), s["b"].data_ptr(), s["d"].data_ptr(),
                                        *ptrs, s["case"]["count"], None, ctypes.byref(worst)), "bcg_muladd_batch_dev")
        return s["c"]
    if kind == "replay":
        s["batch"].run()
        return s["c"]
    if kind == "chain":
        n, bits = s["case"]["points"], s["case"]["bits"]
        a, b, c = s["a"], s["b"], s["c"]
        za, zb = s["za"].data_ptr(), s["zb"].data_ptr()
        pts = ctypes.c_size_t()
        m = ctypes.c_double()
        bc.check(L.bcg_int_to_fft_dev(za, n, a.data_ptr(), a.numel(), bits, ctypes.byref(pts), None), "int_to_fft")
        bc.check(L.bcg_int_to_fft_dev(zb, n, b.data_ptr(), b.numel(), bits, ctypes.byref(pts), None), "int_to_fft")
        bc.check(L.bcg_fft_forward_dev(za, n, None), "fft_forward")
        bc.check(L.bcg_fft_forward_dev(zb, n, None), "fft_forward")
        bc.check(L.bcg_fft_pointwise_dev(za, zb, n, None), "fft_pointwise")
        bc.check(L.bcg_fft_inverse_dev(za, n, None), "fft_inverse")
        bc.check(L.bcg_fft_to_int_dev(za, n, c.data_ptr(), c.numel(), bits, ctypes.byref(m), None), "fft_to_int")
        return {"words": c, "inverse": s["za"], "spectrum_b": s["zb"]}
    if kind == "div":
        bc.bf_op("div", s["t"], s["a"], s["b"], s["case"]["p"])
        words, exp, sign = s["t"].triple()
        return {"words": words, "exp": int(exp), "sign": int(sign)}
    bc.check(L.bcg_radix_dev(s["f"].data_ptr(), s["f"].numel(), s["groups"], s["d"].data_ptr()), "bcg_radix_dev")
    return s["d"]


# --------------------------------------------------------------------- work

def _product_work(al, bl, square=False):
    """Words read and written once; three transforms (two for a square) of the
    al + bl complex points that 16-bit digits of the product take, or the
    word products of the schoolbook method where those are fewer."""
    n = al + bl
    flops = 5.0 * n * max(1.0, math.log2(n)) * (2 if square else 3)
    return 4.0 * ((al if square else al + bl) + n), min(flops, 2.0 * al * bl)


def work(case):
    kind = case["kind"]
    if kind in ("mul", "host"):
        b, f = _product_work(case["al"], case["bl"])
    elif kind == "sqr":
        b, f = _product_work(case["al"], case["al"], True)
    elif kind == "level":
        pl, ql, dl = _level_lengths(case)
        b = f = 0.0
        for x, y, z in zip(pl.tolist(), ql.tolist(), dl.tolist()):
            pb, pf = _product_work(x, y)
            b += pb + 4.0 * z
            f += pf
    elif kind == "replay":
        b = f = 0.0
        for x, y in zip(*(v.tolist() for v in _replay_lengths(case))):
            pb, pf = _product_work(x, y)
            b += pb
            f += pf
    elif kind == "chain":
        n = case["points"]
        w = n * case["bits"] // 64
        b, f = 16.0 * w + 32.0 * n, 15.0 * n * math.log2(n) + 6.0 * n
    elif kind == "div":
        # the last Newton step and the quotient's product: three products of p words
        b, f = _product_work(case["p"], case["p"])
        b, f = 12.0 * case["p"], 3.0 * f
    else:
        # two products of half the length on each of log2(words / 1024) levels of the remainder tree
        n = case["words"]
        levels = max(1.0, math.log2(max(2.0, n / 1024)))
        b, f = 8.0 * n, levels * _product_work(n // 2 + 1, n // 2 + 1)[1]
    return {"bytes": b, "flops": f}


# -------------------------------------------------------------------- exact

def _digits(words, bits, n):
    """The `bits`-bit digits of a word array as float64, padded to n points."""
    b = np.unpackbits(words.view(np.uint8), bitorder="little")
    pts = -(-b.size // bits)
    b = np.concatenate([b, np.zeros(pts * bits - b.size, np.uint8)]).reshape(pts, bits)
    d = b.astype(np.float64) @ (2.0 ** np.arange(bits))
    return np.concatenate([d, np.zeros(n - pts)])


def _order(n):
    """Frequency held at each output place of fft_forward: bit-reversed, with
    the radix-3 digit innermost."""
    p2 = n // 3 if n % 3 == 0 else n
    k = np.zeros(1, dtype=np.int64)
    while k.size < p2:
        k = np.concatenate([2 * k, 2 * k + 1])
    if n % 3 == 0:
        k = (k[:, None] + p2 * np.arange(3, dtype=np.int64)[None, :]).reshape(-1)
    return k


def exact(case, seed):
    if case["kind"] != "chain":
        return None  # whole words: equal or wrong
    n, bits = case["points"], case["bits"]
    w = n * bits // 64
    gen = _gen(seed)
    a = _digits(_words(gen, w).cpu().numpy(), bits, n)
    b = _digits(_words(gen, w).cpu().numpy(), bits, n)
    fa, fb = np.fft.fft(a), np.fft.fft(b)
    # the cyclic product's coefficients are whole numbers far below 2^53
    prod = np.rint(np.fft.ifft(fa * fb).real) * n
    inverse = np.zeros(2 * n)
    inverse[0::2] = prod
    # fft_forward uses e^{+2 pi i / n}: the conjugate of numpy's for real input
    spec = np.conj(fb)[_order(n)]
    return {"words": None, "inverse": torch.from_numpy(inverse),
            "spectrum_b": torch.from_numpy(np.ascontiguousarray(spec).view(np.float64).copy())}
