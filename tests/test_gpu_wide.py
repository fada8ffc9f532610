"""The 16-token half-tile kernel (lw_wide.hip) through the C-ABI, against fp64: every format, the smallest shapes and the
ones that put a row of units into one block, across two and across many, 5..16 tokens of fp16 and 1..8 of fp32
activations, groups of several formats in one call, activations at any alignment, a caller's scratch at its limit, large
and infinite activations and packed twins."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# fp32 sums of exact products, K <= 14336 terms in sums of 16: 2-norm errors of a few 2^-24
TOL = 1e-6
H = {1: 2.3, 2: 3.4, 3: 4.3, 4: 2.6}


def open_mats(tmp_path, mats):
    from lazyweights_amd import Runtime, bundle
    bundle.write_synthetic_bundle(str(tmp_path), mats, threads=16)
    rt = Runtime(tmp_path)
    w = {}
    for name, kqt, N, K, h, seed in mats:
        w[name] = bundle.synth_matrix(kqt, N, K, h, seed, threads=16)
    return rt, w


def y64(orc, kqt, w, x):
    return orc.gemv_f64(orc.dequant(kqt, *w), x.float().cpu().double().numpy())


def err(y, ref):
    y = y.double().cpu().numpy()
    return np.linalg.norm(y - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("kqt", (1, 2, 3, 4))
def test_formats_shapes_and_tokens(gpu, lib, orc, tmp_path, kqt):
    import torch
    cols = 512 if kqt in (1, 4) else 256
    # units per row: 1, 3, 8 (a block holds whole rows), 9 (4-wave blocks, rows shared), 28 in a tall matrix
    mats = [("r%d" % i, kqt, n, k * cols, H[kqt], 900 + i)
            for i, (n, k) in enumerate(((64, 1), (192, 3), (320, 8), (128, 9), (640, 28)))]
    rt, w = open_mats(tmp_path, mats)
    try:
        for name, _, N, K, _, seed in mats:
            for m, f16 in ((5, True), (7, True), (9, True), (16, True), (1, False), (3, False), (8, False)):
                g = torch.Generator().manual_seed(seed + m)
                x = torch.randn(m, K, generator=g)
                x = (x.half() if f16 else x).cuda()
                y = torch.full((m, N + 3), float("nan"), device="cuda")
                for _ in range(2):  # the second call finds slots and counters as the first left them
                    assert lib.lw_matmul_dev(rt.h, name.encode(), x.data_ptr(), int(f16), m, y.data_ptr(), N + 3, None) == 0
                torch.cuda.synchronize()
                e = err(y[:, :N], y64(orc, kqt, w[name], x))
                print(name, kqt, N, K, m, f16, "err %.2g" % e, flush=True)
                assert e < TOL
                assert torch.isnan(y[:, N:]).all()
    finally:
        rt.close()


def test_group_of_formats_and_alignment(gpu, lib, orc, tmp_path):
    import torch
    mats = [("a", 1, 256, 4096, H[1], 1), ("b", 3, 128, 4096, H[3], 2), ("c", 2, 192, 1024, H[2], 3),
            ("d", 4, 64, 4096, H[4], 4)] + [("e%d" % i, 1 + i % 4, 64, 1024, H[1 + i % 4], 5 + i) for i in range(6)]
    rt, w = open_mats(tmp_path, mats)
    try:
        for m, shift in ((6, 0), (16, 1), (7, 4)):  # x shared by equal K, `shift` fp16 past a 16-byte boundary
            xs = {}
            for K in (1024, 4096):
                buf = torch.zeros(m * K + 8, dtype=torch.float16, device="cuda")
                buf[shift:shift + m * K] = torch.randn(m * K, generator=torch.Generator().manual_seed(m + K)).half().cuda()
                xs[K] = buf[shift:shift + m * K].view(m, K)
            ys = [torch.zeros(m, mat[2], device="cuda") for mat in mats]
            n = len(mats)
            assert lib.lw_group_matmul_dev(rt.h, n, (ctypes.c_char_p * n)(*[mt[0].encode() for mt in mats]),
                                           (ctypes.c_void_p * n)(*[xs[mt[3]].data_ptr() for mt in mats]), m,
                                           (ctypes.c_void_p * n)(*[y.data_ptr() for y in ys]), None) == 0
            torch.cuda.synchronize()
            for mt, y in zip(mats, ys):
                assert err(y, y64(orc, mt[1], w[mt[0]], xs[mt[3]])) < TOL, (mt, m, shift)
    finally:
        rt.close()


def test_token_order_nan_and_scratch_limit(gpu, lib, orc, tmp_path):
    """A NaN token leaves the others their bits and the partial slots consistent; without allocation the reordered
    activations go into the partials' tail where the 16 MiB hold no more (16 x 8 x 32768 partials are exactly that less
    the counters, so 32256 rows are the most)."""
    import torch
    mats = [("m", 1, 32256, 4096, 2.3, 11), ("s", 1, 128, 4608, 2.3, 12)]
    rt, w = open_mats(tmp_path, mats)
    try:
        K = 4096
        x = torch.randn(16, K, generator=torch.Generator().manual_seed(3)).half().cuda()
        ya, yb = (torch.zeros(16, 32256, device="cuda") for _ in range(2))
        for fn, y in ((lib.lw_matmul_dev, ya), (lib.lw_matmul_dev_noalloc, yb)):
            assert fn(rt.h, b"m", x.data_ptr(), 1, 16, y.data_ptr(), 32256, None) == 0, lib.lw_last_error()
        torch.cuda.synchronize()
        assert torch.equal(ya, yb)
        assert err(ya, y64(orc, 1, w["m"], x)) < TOL
        x = torch.randn(9, 4608, generator=torch.Generator().manual_seed(4)).half().cuda()
        ref, y = (torch.zeros(9, 128, device="cuda") for _ in range(2))
        lib.lw_matmul_dev(rt.h, b"s", x.data_ptr(), 1, 9, ref.data_ptr(), 128, None)
        bad = x.clone()
        bad[4, 100] = float("nan")
        lib.lw_matmul_dev(rt.h, b"s", bad.data_ptr(), 1, 9, y.data_ptr(), 128, None)
        torch.cuda.synchronize()
        keep = [i for i in range(9) if i != 4]
        assert torch.isnan(y[4]).all() and torch.equal(y[keep], ref[keep])
        lib.lw_matmul_dev(rt.h, b"s", x.data_ptr(), 1, 9, y.data_ptr(), 128, None)
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
    finally:
        rt.close()


@pytest.mark.parametrize("kqt", (1, 2))
def test_sub_block_sums_past_fp16(gpu, lib, orc, tmp_path, kqt):
    """The mins take the sums of 32 activations in the range and with the bits of fp32: sub-blocks of 3000 (a sum of 96000,
    past fp16's largest number), two activations of 40000, and 32 of the largest fp16 number, beside ordinary ones. Measured
    against sum |w x|, the size of the terms: fp32 sums of 16, so a few 2^-24."""
    import torch
    rt, w = open_mats(tmp_path, [("a", kqt, 192, 4608, H[kqt], 31)])
    try:
        d = orc.dequant(kqt, *w["a"])
        for m, f16 in ((1, True), (5, True), (9, True), (16, True), (1, False), (8, False)):
            x = torch.randn(m, 4608, generator=torch.Generator().manual_seed(m))
            x[0, 96:128] = 3000
            x[m // 2, [512, 540]] = 40000
            x[m - 1, 4576:] = -65504
            x = (x.half() if f16 else x).cuda()
            y = torch.full((m, 192), float("nan"), device="cuda")
            assert lib.lw_matmul_dev(rt.h, b"a", x.data_ptr(), int(f16), m, y.data_ptr(), 192, None) == 0
            torch.cuda.synchronize()
            y = y.double().cpu().numpy()
            x64 = x.float().cpu().double().numpy()
            ref, size = orc.gemv_f64(d, x64), orc.gemv_f64(np.abs(d), np.abs(x64))
            e = np.linalg.norm(y - ref, axis=1) / np.linalg.norm(size, axis=1)
            print("sums", kqt, m, f16, "err %.2g" % e.max(), flush=True)
            assert e.max() < TOL, (m, f16)
    finally:
        rt.close()


@pytest.mark.parametrize("kqt", (1, 2, 3, 4))
def test_packed_twin_and_host_entry(gpu, lib, orc, tmp_path, kqt):
    """A packed twin gives the coded matrix's bits with fp32 activations and with 9..16 tokens of fp16 (row units: 1, 8 in one
    block, 9 over several), alone and grouped over two formats; rt_test_matmul gives lw_matmul_dev's."""
    import torch
    from lazyweights_amd import Runtime, bundle
    cols = 512 if kqt in (1, 4) else 256
    mats = [("r%d" % i, kqt, n, k * cols, H[kqt], 950 + i) for i, (n, k) in enumerate(((64, 1), (192, 8), (128, 9)))]
    mats.append(("o", kqt % 4 + 1, 64, 9 * 512, H[kqt % 4 + 1], 960))
    bundle.write_synthetic_bundle(str(tmp_path / "coded"), mats, threads=16)
    bundle.write_packed_bundle(str(tmp_path / "packed"), mats, threads=16)
    with Runtime(tmp_path / "coded") as rc, Runtime(tmp_path / "packed") as rp:
        for name, kq, N, K, _, seed in mats:
            w = bundle.synth_matrix(kq, N, K, H[kq], seed, threads=16)
            for m, f16 in ((1, False), (3, False), (8, False), (9, True), (16, True)):
                x = torch.randn(m, K, generator=torch.Generator().manual_seed(seed + m))
                x = (x.half() if f16 else x).cuda()
                yc, yp = (torch.full((m, N), float("nan"), device="cuda") for _ in range(2))
                rc.matmul_dev(name, x, yc, x_f16=f16)
                for _ in range(2):
                    rp.matmul_dev(name, x, yp, x_f16=f16)
                torch.cuda.synchronize()
                assert torch.equal(yc, yp), (name, m, f16)
                assert err(yp, y64(orc, kq, w, x)) < TOL, (name, m, f16)
                if not f16:
                    for rt in (rc, rp):
                        assert np.array_equal(rt.test_matmul(name, x.cpu().numpy()), yc.cpu().numpy()), (name, m)
        n, xs = len(mats), [torch.randn(11, m[3], generator=torch.Generator().manual_seed(m[3])).half().cuda() for m in mats]
        ys = []
        for rt in (rc, rp):
            ys.append([torch.zeros(11, m[2], device="cuda") for m in mats])
            assert lib.lw_group_matmul_dev(rt.h, n, (ctypes.c_char_p * n)(*[m[0].encode() for m in mats]),
                                           (ctypes.c_void_p * n)(*[x.data_ptr() for x in xs]), 11,
                                           (ctypes.c_void_p * n)(*[y.data_ptr() for y in ys[-1]]), None) == 0
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(*ys))


@pytest.mark.parametrize("kqt", (3, 4))
def test_infinite_activation(gpu, lib, orc, tmp_path, kqt):
    """An infinite fp16 activation gives infinities of its products' signs in Q6_K and IQ4_XS, which have no mins (and NaN
    where the weight is 0), and leaves the other tokens alone."""
    import torch
    rt, w = open_mats(tmp_path, [("a", kqt, 128, 4608, H[kqt], 33)])
    try:
        d = orc.dequant(kqt, *w["a"])
        for m in (5, 9, 16):
            x = torch.randn(m, 4608, generator=torch.Generator().manual_seed(m)).half()
            x[1, 700], x[m - 1, 4000] = float("inf"), float("-inf")
            y = torch.zeros(m, 128, device="cuda")
            xd = x.cuda()
            assert lib.lw_matmul_dev(rt.h, b"a", xd.data_ptr(), 1, m, y.data_ptr(), 128, None) == 0
            torch.cuda.synchronize()
            y = y.cpu().numpy()
            with np.errstate(invalid="ignore"):
                for tok, col, sign in ((1, 700, 1), (m - 1, 4000, -1)):
                    want = sign * np.inf * d[:, col]
                    print("inf", kqt, m, int(np.isinf(y[tok]).sum()), "of", int(np.isinf(want).sum()), flush=True)
                    assert np.array_equal(y[tok], want, equal_nan=True), (m, tok)
            keep = [t for t in range(m) if t not in (1, m - 1)]
            assert err(torch.from_numpy(y[keep]), y64(orc, kqt, w["a"], x[keep])) < TOL
    finally:
        rt.close()


@pytest.mark.parametrize("kqt", (2, 3))
def test_short_sums_no_further_than_the_4_token_kernel(gpu, lib, orc, tmp_path, kqt):
    """The 8-bit formats over few super-blocks, where a product's rounding shows: 16 tokens in one call are as near to fp64
    as the same ones four by four, which the whole-tile kernel sums in integers scaled per sub-block. (Roundings of another
    order on 16 x 1024 results: 2 % either way.)"""
    import torch
    rt, w = open_mats(tmp_path, [("k%d" % k, kqt, 1024, k, H[kqt], 70 + k) for k in (256, 512, 768, 1024)])
    try:
        for name in w:
            K = int(name[1:])
            x = torch.randn(16, K, generator=torch.Generator().manual_seed(K)).half().cuda()
            y, y4 = (torch.zeros(16, 1024, device="cuda") for _ in range(2))
            rt.matmul_dev(name, x, y)
            for t in range(0, 16, 4):
                rt.matmul_dev(name, x[t:t + 4], y4[t:t + 4])
            torch.cuda.synchronize()
            ref = y64(orc, kqt, w[name], x)
            print("short", kqt, K, "%.3g %.3g" % (err(y, ref), err(y4, ref)), flush=True)
            assert err(y, ref) <= 1.02 * err(y4, ref), K
    finally:
        rt.close()


@pytest.mark.parametrize("kqt", (1, 2, 3, 4))
def test_block_sizes_and_uneven_tiles(gpu, lib, orc, tmp_path, kqt):
    """Rows of 6 units (whole, blocks of 6 waves), of 2 and 3 where blocks of 8 waves are at most one per CU and blocks of 4
    more (a last block with rows left over), and tiles whose halves and rows differ in length: runs of the most frequent
    code beside uniform codes."""
    import torch
    from lazyweights_amd import Runtime
    from lazyweights_amd.bundle import Writer, synth_matrix
    cols, ncodes = (512, 16) if kqt in (1, 4) else (256, 32 if kqt == 2 else 64)
    rng = np.random.default_rng(kqt)
    w, out = Writer(str(tmp_path)), {}
    for name, N, units in (("six", 192, 6), ("two", 64 * 301, 2), ("three", 64 * 151, 3), ("uneven", 256, 9)):
        codes, side = synth_matrix(kqt, N, units * cols, H[kqt], 80 + units, threads=16)
        if name == "uneven":
            codes[:] = ncodes // 2
            for r0 in (0, 40, 96, 128, 200):  # 8 to 32 long rows in the one half or the other, the rest a bit per symbol
                codes[r0:r0 + 8 + r0 % 25] = rng.integers(0, ncodes, (8 + r0 % 25, units * cols))
        w.add_kquant(name, kqt, codes, side)
        out[name] = (codes, side)
    w.close()
    with Runtime(tmp_path) as rt:
        for name, (codes, side) in out.items():
            N, K = codes.shape
            d = orc.dequant(kqt, codes, side).astype(np.float64)
            for m, f16 in ((5, True), (16, True), (3, False)):
                x = torch.randn(m, K, generator=torch.Generator().manual_seed(m))
                x = (x.half() if f16 else x).cuda()
                y = torch.full((m, N), float("nan"), device="cuda")
                for _ in range(2):
                    rt.matmul_dev(name, x, y, x_f16=f16)
                torch.cuda.synchronize()
                ref = x.double().cpu().numpy() @ d.T
                e = err(y, ref)
                print("blocks", name, kqt, N, K, m, f16, "err %.2g" % e, flush=True)
                assert e < TOL, (name, m)


@pytest.mark.parametrize("ends", ("low", "high", "zeros"))
def test_one_sided_codes(gpu, lib, orc, tmp_path, ends):
    """Q5_K codes that lie at an end of their range: what the kernel takes off every code follows them (16 for all of them
    put such results up to 25 times as far from fp64 as the 4-token kernel's), and a packed twin, whose codes are the same,
    has the bits. Bound, in squares of a rounding at the result's size: a unit's one run of 16 additions rounds 1/16 + .. +
    16/16 = 8.5, where the rest of the codes makes up the whole result, its fold and sums 3; the 4-token kernel's 8 folds
    per super-block 4.5 and its sum 1: the square root of 11.5 / 5.5 is 1.45."""
    import torch
    from lazyweights_amd import Runtime
    from lazyweights_amd.bundle import Writer, synth_matrix
    rng = np.random.default_rng(9)
    out = {}
    for d in ("coded", "packed"):
        w = Writer(str(tmp_path / d))
        for K in (1024, 4096):
            if d == "coded":
                _, side = synth_matrix(2, 512, K, H[2], 90, threads=16)
                codes = np.minimum(rng.geometric(0.8 if ends == "zeros" else 0.35, (512, K)) - 1, 31).astype(np.uint8)
                out[K] = (31 - codes if ends == "high" else codes, side)
            w.add_kquant("k%d" % K, 2, *out[K], packed=d == "packed")
        w.close()
    with Runtime(tmp_path / "coded") as rc, Runtime(tmp_path / "packed") as rp:
        for K in out:
            x = torch.randn(16, K, generator=torch.Generator().manual_seed(K)).half().cuda()
            y, y4, yp = (torch.zeros(16, 512, device="cuda") for _ in range(3))
            rc.matmul_dev("k%d" % K, x, y)
            rp.matmul_dev("k%d" % K, x, yp)
            for t in range(0, 16, 4):
                rc.matmul_dev("k%d" % K, x[t:t + 4], y4[t:t + 4])
            torch.cuda.synchronize()
            ref = y64(orc, 2, out[K], x)
            print("one-sided", ends, K, "%.3g %.3g" % (err(y, ref), err(y4, ref)), flush=True)
            assert err(y, ref) <= 1.45 * err(y4, ref), K
            assert torch.equal(y, yp)
