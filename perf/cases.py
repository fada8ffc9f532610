"""The work a program has this library do, for timing: GEMVs and skinny GEMMs of a decoder layer's coded matrices at
every batch the entry points take, prefill GEMMs, int8 activations, and GPU decode to codes.

A case names its matrices ("Q4_K:4096x4096:2.3" is format, N x K and entropy in bits per code), which of them share
one call ("0 1 2|3|4 5|6": the matrices of a group that have the same K take the same activations, as q, k, v or gate
and up do, and a group depends on the one before it in a forward pass), the token count m, the activations' type, and
whether they are quantized to int8. Shapes and entropies are those of lazyweights_amd/configs.py. Weights are drawn as there: codes
from a two-sided geometric distribution of the given entropy, d and dmin uniform in [0.005, 0.02], 6-bit sub-scales
(int8 for Q6_K) uniform; activations are normal.
"""
import ctypes
import math
import tempfile

import numpy as np
import torch

from lazyweights_amd import Runtime, bundle

NCODES = {"Q4_K": 16, "Q5_K": 32, "Q6_K": 64, "IQ4_XS": 16}
ENTROPY = {"Q4_K": 2.3, "Q5_K": 3.4, "Q6_K": 4.3, "IQ4_XS": 2.6}
SIDE = {"Q4_K": 16, "Q5_K": 16, "Q6_K": 18, "IQ4_XS": 8}  # bytes per 256 weights
IQ4_GRID = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
MISTRAL = "{f}:4096x4096:{e},{f}:1024x4096:{e},{f}:1024x4096:{e},{f}:4096x4096:{e}," \
          "{f}:14336x4096:{e},{f}:14336x4096:{e},{f}:4096x14336:{e}"
FORWARD = "0 1 2|3|4 5|6"


def listed():
    q4, q5 = MISTRAL.format(f="Q4_K", e=2.3), MISTRAL.format(f="Q5_K", e=3.4)
    return [
        # one token through one small projection: the smallest call, launch latency
        {"name": "k projection m=1", "mats": "Q4_K:1024x4096:2.3", "groups": "0", "m": 1, "x": "f16", "do": "mul"},
        # one token through a small model's layer, a call per dependent step of the forward pass
        {"name": "phi layer m=1", "mats": "Q4_K:9216x3072:2.6,Q4_K:3072x3072:2.6,Q4_K:16384x3072:2.6,Q4_K:3072x8192:2.6",
         "groups": "0|1|2|3", "m": 1, "x": "f16", "do": "mul"},
        # a whole layer's matrices in one grouped call: the benchmark's headline unit
        {"name": "mistral layer grouped m=1", "mats": q4, "groups": "0 1 2 3 4 5 6", "m": 1, "x": "f16", "do": "mul"},
        # speculative verification of 5 tokens, mixed formats
        {"name": "mixed mlp verify m=5", "mats": "Q6_K:4096x14336:4.3,IQ4_XS:14336x4096:2.6,IQ4_XS:14336x4096:2.6",
         "groups": "1 2|0", "m": 5, "x": "f16", "do": "mul"},
        # 16 sequences decoded together
        {"name": "mistral layer batch m=16", "mats": q4, "groups": FORWARD, "m": 16, "x": "f16", "do": "mul"},
        # int8 activations, one token
        {"name": "mistral layer int8 m=1", "mats": q5, "groups": FORWARD, "m": 1, "x": "f16", "do": "int8"},
        # fp32 activations of a short draft: a program that keeps its hidden state in fp32
        {"name": "phi layer f32 m=4", "mats": "Q4_K:9216x3072:2.6,Q4_K:3072x3072:2.6,Q4_K:16384x3072:2.6,Q4_K:3072x8192:2.6",
         "groups": "0|1|2|3", "m": 4, "x": "f32", "do": "mul"},
        # a short prompt of an odd length
        {"name": "iq4 gate prompt m=33", "mats": "IQ4_XS:14336x4096:2.6", "groups": "0", "m": 33, "x": "f32", "do": "mul"},
        # a prompt chunk through a whole layer
        {"name": "mistral layer prompt m=128", "mats": q4, "groups": FORWARD, "m": 128, "x": "f32", "do": "mul"},
        # a prompt through the widest reduction
        {"name": "q6 down prompt m=512", "mats": "Q6_K:4096x14336:4.3", "groups": "0", "m": 512, "x": "f32", "do": "mul"},
        # a long prompt: the largest call
        {"name": "q4 gate prompt m=2048", "mats": "Q4_K:14336x4096:2.3", "groups": "0", "m": 2048, "x": "f32", "do": "mul"},
        # decode to host codes, a byte per weight (checking or converting a bundle)
        {"name": "codes 4096x4096", "mats": "Q4_K:4096x4096:2.6", "groups": "0", "m": 1, "x": "f16", "do": "codes"},
    ]


def _spread(rng, low, high):
    """A whole number in low .. high, uniform over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    fmt = rng.choice(sorted(NCODES))
    e = round(ENTROPY[fmt] + rng.uniform(-0.2, 0.3), 2)
    n, k = 64 * _spread(rng, 4, 256), 512 * _spread(rng, 1, 28)
    if NCODES[fmt] > 16 and rng.random() < 0.5:
        k += 256
    mats, groups = "%s:%dx%d:%s" % (fmt, n, k, e), "0"
    do, x = rng.choice((("mul", "f16"), ("mul", "f16"), ("mul", "f32"), ("mul", "f32"), ("mul", "prompt"), ("mul", "prompt"),
                        ("int8", "f16"), ("codes", "f16")))
    if x == "f16":
        m = _spread(rng, 1, 8 if do == "int8" else 16) if do != "codes" else 1
        if do != "codes" and rng.random() < 0.5:  # a second and a third matrix of the same activations
            mats += ",%s:%dx%d:%s,%s:%dx%d:%s" % (fmt, 64 * _spread(rng, 4, 128), k, e, fmt, 64 * _spread(rng, 4, 128), k, e)
            groups = "0 1 2"
    else:
        m, x = (_spread(rng, 1, 8) if x == "f32" else _spread(rng, 9, 2048)), "f32"
        m = max(1, min(m, 2048 * 14336 * 4096 // (n * k)))
    return {"mats": mats, "groups": groups, "m": m, "x": x, "do": do}


def _mats(case):
    out = []
    for text in case["mats"].split(","):
        fmt, shape, e = text.split(":")
        n, k = shape.split("x")
        out.append((fmt, int(n), int(k), float(e)))
    return out


def _groups(case):
    return [[int(i) for i in g.split()] for g in case["groups"].split("|")]


def _code_table(fmt, entropy):
    """65536 codes: entry u is the code of the uniform 16-bit number u (two-sided geometric of the given entropy)."""
    nc = NCODES[fmt]
    off = np.abs(np.arange(nc) - nc // 2)
    low, high = 1e-6, 1 - 1e-9
    for _ in range(60):
        rho = (low + high) / 2
        p = rho ** off
        p /= p.sum()
        low, high = (rho, high) if -(p * np.log2(np.maximum(p, 1e-300))).sum() < entropy else (low, rho)
    cum = np.cumsum(p)
    return np.minimum(np.searchsorted(cum, (np.arange(65536) + 0.5) / 65536), nc - 1).astype(np.uint8)


def _weights(fmt, n, k, entropy, seed):
    """codes [n, k] and side records [n, k / 256, bytes], uint8 on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    table = torch.from_numpy(_code_table(fmt, entropy)).cuda()
    codes = table[torch.randint(0, 65536, (n, k), generator=g, device="cuda")]
    nb = k // 256
    scale = [(torch.rand((n, nb, 1), generator=g, device="cuda") * 0.015 + 0.005).half().view(torch.uint8) for _ in range(2)]
    r = torch.randint(0, 256, (n, nb, 16), generator=g, device="cuda")
    if fmt == "Q6_K":
        side = [((r % 255) - 127).to(torch.int8).view(torch.uint8), scale[0]]
    elif fmt == "IQ4_XS":
        side = [scale[0], r[..., :6].to(torch.uint8)]
    else:
        side = [scale[0], scale[1], r[..., :12].to(torch.uint8)]
    return codes, torch.cat(side, dim=2).contiguous()


def _inputs(case, seed):
    """The matrices, their weights and each matrix's activations [m, K] (one tensor per group and K)."""
    mats = _mats(case)
    w = [_weights(*mat, seed * 64 + i) for i, mat in enumerate(mats)]
    g = torch.Generator(device="cuda").manual_seed(seed * 64 + 63)
    xs = [None] * len(mats)
    for group in _groups(case):
        shared = {}
        for i in group:
            k = mats[i][2]
            if k not in shared:
                x = torch.randn((case["m"], k), generator=g, device="cuda")
                shared[k] = x.half() if case["x"] == "f16" else x
            xs[i] = shared[k]
    return mats, w, xs


def prepare(case, seed):
    mats, w, xs = _inputs(case, seed)
    with tempfile.TemporaryDirectory() as d:
        out = bundle.Writer(d)
        for i, ((fmt, n, k, _), (codes, side)) in enumerate(zip(mats, w)):
            pairs = bundle.SYMBITS[bundle.KQ[fmt]] == 4
            sym = codes[:, 0::2] | (codes[:, 1::2] << 4) if pairs else codes
            blob, _ = bundle.encode_huf8(sym.cpu().numpy())
            out.add("w%d" % i, "huf4p" if pairs else "huf8", n, k, 1.0, 0, blob)
            out.add("w%d.kqs" % i, "kq_" + fmt, n, side.shape[1] * side.shape[2], 1.0, 0, side.cpu().numpy().tobytes())
        out.close()
        rt = Runtime(d)
    calls = []
    for group in _groups(case):
        x = [xs[i] for i in group]
        ys = [torch.zeros((case["m"], mats[i][1]), device="cuda") for i in group]
        for i, xi, y in zip(group, x, ys):  # the library takes bare pointers
            if (rt.info("w%d" % i)["N"], rt.info("w%d" % i)["K"]) != (y.shape[1], xi.shape[1]) or not xi.is_contiguous():
                raise ValueError("w%d: activations %s, outputs %s" % (i, tuple(xi.shape), tuple(y.shape)))
        names = (ctypes.c_char_p * len(group))(*[b"w%d" % i for i in group])
        xp = (ctypes.c_void_p * len(group))(*[xi.data_ptr() for xi in x])
        yp = (ctypes.c_void_p * len(group))(*[y.data_ptr() for y in ys])
        calls.append((group, x, ys, names, xp, yp))
    return {"rt": rt, "lib": rt.lib, "do": case["do"], "m": case["m"], "f16": case["x"] == "f16", "calls": calls}


def run(state):
    rt, lib, f16 = state["rt"], state["lib"], state["f16"]
    if state["do"] == "codes":
        return rt.test_decode("w0")
    if state["do"] == "int8":
        lib.lw_set_act8(1)
    try:
        for group, x, ys, names, xp, yp in state["calls"]:
            if f16 and len(group) > 1:
                if lib.lw_group_matmul_dev(rt.h, len(group), names, xp, state["m"], yp, None) != 0:
                    raise RuntimeError(lib.lw_last_error().decode())
            else:
                for i, xi, y in zip(group, x, ys):
                    rt.matmul_dev("w%d" % i, xi, y, x_f16=f16)
    finally:
        if state["do"] == "int8":
            lib.lw_set_act8(0)
    return [y for call in state["calls"] for y in call[2]]


def work(case):
    """Coded words at the codes' entropy, side records, activations once per group, outputs."""
    mats = _mats(case)
    total = sum(n * k * e / 8 + n * k // 256 * SIDE[fmt] for fmt, n, k, e in mats)
    if case["do"] == "codes":
        fmt, n, k, e = mats[0]
        return {"bytes": n * k * e / 8 + n * k, "flops": 0}
    size = 2 if case["x"] == "f16" else 4
    total += sum(size * case["m"] * k for g in _groups(case) for k in {mats[i][2] for i in g})
    total += sum(4 * case["m"] * n for _, n, _, _ in mats)
    return {"bytes": total, "flops": sum(2 * case["m"] * n * k for _, n, k, _ in mats)}


def tolerance(case):
    if case["do"] == "codes":
        return "exact"
    # fp32 sums of exact products, in any order; about four times the distance from 64 bits measured on MI355X: 2e-7 at
    # most for int8 activations and prompts, 9e-6 where up to 16 tokens of a 4-bit format with mins go through fp16 dot
    # products (the terms with and without the mins cancel to a tenth)
    return {"rel": 1e-6 if case["do"] == "int8" or case["m"] > 16 or (case["x"] == "f32" and case["m"] > 8) else 4e-5}


def _dequantized(fmt, codes, side):
    """Weights [n, k] in 64 bits, llama.cpp's block semantics."""
    n, k = codes.shape
    s = side.to(torch.int64)

    def half(i):
        return side[..., i:i + 2].contiguous().view(torch.float16).double()

    if fmt == "Q6_K":
        sub = side[..., :16].contiguous().view(torch.int8).double() * half(16)
        return (codes.double().sub_(32).view(n, k // 256, 16, 16) * sub[..., None]).view(n, k)
    if fmt == "IQ4_XS":
        hi = s[..., 2] | (s[..., 3] << 8)
        ls = torch.stack([((s[..., 4 + j // 2] >> (4 * (j % 2))) & 15) | (((hi >> (2 * j)) & 3) << 4) for j in range(8)], -1)
        grid = torch.tensor(IQ4_GRID, dtype=torch.float64, device="cuda")
        return (grid[codes.long()].view(n, k // 256, 8, 32) * ((ls - 32).double() * half(0))[..., None]).view(n, k)
    a, b, c = s[..., 4:8], s[..., 8:12], s[..., 12:16]
    sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], -1).double() * half(0)
    mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], -1).double() * half(2)
    return (codes.double().view(n, k // 256, 8, 32) * sc[..., None] - mn[..., None]).view(n, k)


def _quantized(x):
    """x as int8 activations stand for it: per block of 32, d = max|x| / 127 in fp32 and d round(x / d)."""
    b = x.float().view(x.shape[0], -1, 32)
    d = b.abs().amax(2, keepdim=True) / 127
    q = torch.where(d > 0, torch.round(b / torch.where(d > 0, d, torch.ones_like(d))), torch.zeros_like(b))
    return (q.double() * d.double()).view(x.shape)


def exact(case, seed):
    mats, w, xs = _inputs(case, seed)
    if case["do"] == "codes":
        return w[0][0].cpu().numpy()
    out = []
    for i in (i for group in _groups(case) for i in group):
        x = _quantized(xs[i]) if case["do"] == "int8" else xs[i].double()
        (codes, side), w[i] = w[i], None
        out.append(x @ _dequantized(mats[i][0], codes, side).T)
    return out
