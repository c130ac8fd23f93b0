"""The column kernels (rq_cols_*, rq_colsglu_*): matvecs over more than 8
Q8_1 columns, and the dot4 layout's fused gate/up from 9, against the integer
oracle at the edges of their tiles, column groups and rows."""
import numpy as np
import pytest
import torch

from gpu_util import make_weight, q8_1_to_device, upload
from rllm_amd.backend import Activation

pytestmark = pytest.mark.gpu

TYPES = {"Q4_0": 2, "Q8_0": 8, "Q4_K": 12, "Q6_K": 14}

# f32 sums over exact products: a row of S super-blocks passes at most 4 + 1
# roundings per half super-block, 2 ceil(S / 8) partial sums and 3 levels of
# eight parts, each 2^-24 of a partial sum. Partial sums of N(0, 1) terms stay
# within about the row's norm, so 1e-5 of the largest output (170 roundings,
# all one way) is out of reach for the widths here.
TOL = 1e-5


def _q8(orc, seed, m, k):
    return orc.quantize_q8_1(orc.normal(seed, m * k, 0.0, 1.0), m, k)


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("n,k", [(1, 256), (16, 512), (17, 2048), (63, 2304), (96, 4096), (33, 13824), (37, 16896),
                                 (40, 32), (24, 160), (50, 2080)])
@pytest.mark.parametrize("m", [9, 16, 17, 43, 64, 70])
def test_cols_matvec(gpu, orc, tname, n, k, m):
    """Both layouts against the oracle, and bit-identical to each other
    wherever both run the column kernels (m > 16, or wide rows): the order of
    the sums depends on the width alone."""
    t = TYPES[tname]
    if t in (12, 14) and k % 256:
        pytest.skip("K-quants need k % 256 == 0")
    w = make_weight(orc, t, n, k, 40 + n, "random")
    qs, d, s = _q8(orc, 41 + k + m, m, k)
    want = orc.matvec_q8_1(t, w, n, k, qs, d, m)
    got = {}
    for fam in ("dot4", "mfma"):
        gpu.set_kernels(fam)
        wg = upload(gpu, t, w, n, k)
        gpu.set_kernels("auto")
        out = gpu.alloc(m * n + 8)
        out.fill_(float("nan"))
        gpu.matvec(q8_1_to_device(gpu, qs, d, s), wg, out, m)
        got[fam] = gpu.to_host(out)
        assert np.isnan(got[fam][m * n:]).all(), "wrote past the output"
        orc.assert_close(f"{tname} {n}x{k} m={m} {fam}", want, got[fam][:m * n], TOL if m > 16 or fam == "dot4" else 1e-3)
    if m > 16:
        assert np.array_equal(got["dot4"][:m * n].view(np.uint32), got["mfma"][:m * n].view(np.uint32))


@pytest.mark.parametrize("tname", list(TYPES))
def test_cols_do_not_depend_on_the_count(gpu, orc, tname):
    """The first columns of a 70-column call (two launches) as calls of 9 and
    33, and of rows enough for two and four tiles per workgroup."""
    t, k = TYPES[tname], 1024
    for n in (40, 16 * 400, 16 * 800):
        w = orc.random_weight(50, t, n, k)
        wg = upload(gpu, t, w, n, k)
        qs, d, s = _q8(orc, 51, 70, k)
        outs = {}
        for m in (70, 33, 9):
            out = gpu.alloc(m * n)
            xq = q8_1_to_device(gpu, qs[:m * k], d[:m * k // 32], s[:m * k // 32])
            gpu.matvec(xq, wg, out, m)
            outs[m] = gpu.to_host(out, m * n).view(np.uint32)
        for m in (33, 9):
            assert np.array_equal(outs[m], outs[70][:m * n]), f"n={n} m={m}"
        rows = np.r_[0:20, n - 20:n]
        want = orc.matvec_q8_1(t, w, n, k, qs[:9 * k], d[:9 * k // 32], 9).reshape(9, n)
        orc.assert_close(f"{tname} {n}x{k}", want[:, rows].reshape(-1),
                         outs[9].view(np.float32).reshape(9, n)[:, rows].reshape(-1), TOL)


@pytest.mark.parametrize("family", ["dot4", "mfma"])
@pytest.mark.parametrize("k", [4096, 13824])
def test_cols_mixed_launch(gpu, orc, family, k):
    """Q4_K and Q6_K weights together are bit-identical to their own calls,
    whichever of them run the column kernels (MFMA: Q6_K does at 20 columns,
    a Q4_K weight of more than 512 tiles does not)."""
    m = 20
    spec = [(12, 48), (14, 33), (12, 8208 if k == 4096 else 17)]
    ws = [orc.random_weight(60 + i, t, n, k) for i, (t, n) in enumerate(spec)]
    gpu.set_kernels(family)
    wgs = [upload(gpu, t, w, n, k) for (t, n), w in zip(spec, ws)]
    gpu.set_kernels("auto")
    x = gpu.from_host(orc.normal(61, m * k, 0.0, 1.0))
    outs = [gpu.alloc(m * n) for _, n in spec]
    gpu.matmul_many(x, wgs, outs, m)
    for (t, n), wg, out in zip(spec, wgs, outs):
        own = gpu.alloc(m * n)
        gpu.matmul(x, wg, own, m)
        assert torch.equal(own.view(torch.int32), out.view(torch.int32)), f"type {t} rows {n}"


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("f,d", [(32, 512), (96, 4096), (64, 5120)])
@pytest.mark.parametrize("m", [8, 9, 16, 17, 33, 50])
def test_cols_gated_ffn(gpu, orc, tname, f, d, m):
    """The dot4 layout's fused front half: h within 1e-3 of the integer path
    (the activation's expf), the down projection on exactly h's Q8_1."""
    t = TYPES[tname]
    gw, uw = orc.random_weight(70, t, f, d), orc.random_weight(71, t, f, d)
    g, u = upload(gpu, t, gw, f, d), upload(gpu, t, uw, f, d)
    qs, dq, s = _q8(orc, 73 + m, m, d)
    h = gpu.alloc(m * f)
    out = gpu.alloc(m * 256)
    down = upload(gpu, 8, orc.random_weight(74, 8, 256, f), 256, f)
    gpu.gated_ffn_q8_1(q8_1_to_device(gpu, qs, dq, s), g, u, down, Activation.SILU, out, h, gpu.alloc(m * f), m)
    orc.assert_close(f"h {tname} {f}x{d} m={m}", orc.glu_q8_1(t, gw, uw, f, d, qs, dq, m, 0), gpu.to_host(h, m * f), 1e-3)
    want = gpu.alloc(m * 256)
    gpu.matvec(gpu.quantize_q8_1(h, m, f), down, want, m)
    assert torch.equal(out.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("n,k", [(9216, 512), (16400, 512), (8208, 1024), (20480, 2304), (8208, 4352), (8240, 2048)])
@pytest.mark.parametrize("m", [17, 32, 41, 49, 64])
def test_q6_k_rows_that_keep_the_int8_classes(gpu, orc, n, k, m):
    """MFMA-layout Q6_K where the int8 classes take fewer rounds (short rows
    of more than 512 tiles, and where three or five tiles fit a workgroup):
    columns as in an 8-column launch, bit for bit, and within 1e-3 of the
    oracle."""
    if m == 41 and 1024 <= k <= 2048:
        pytest.skip("the column kernels' at 33 to 48 columns")
    t = TYPES["Q6_K"]
    w = orc.random_weight(90, t, n, k)
    gpu.set_kernels("mfma")
    wg = upload(gpu, t, w, n, k)
    gpu.set_kernels("auto")
    qs, d, s = _q8(orc, 91 + m, m, k)
    out, eight = gpu.alloc(m * n), gpu.alloc(8 * n)
    gpu.matvec(q8_1_to_device(gpu, qs, d, s), wg, out, m)
    for c0 in (0, 8, m - 8):
        part = q8_1_to_device(gpu, qs[c0 * k:(c0 + 8) * k], d[c0 * k // 32:(c0 + 8) * k // 32], s[c0 * k // 32:(c0 + 8) * k // 32])
        gpu.matvec(part, wg, eight, 8)
        assert torch.equal(out[c0 * n:(c0 + 8) * n], eight[:8 * n]), f"columns {c0}.."
    rows = np.r_[0:17, n - 17:n]
    rb = w.reshape(n, -1)
    want = orc.matvec_q8_1(t, np.ascontiguousarray(rb[rows]).reshape(-1), len(rows), k, qs, d, m)
    got = gpu.to_host(out, m * n).reshape(m, n)[:, rows].reshape(-1)
    orc.assert_close(f"Q6_K {n}x{k} m={m}", want, got, 1e-3)


# Rows for two and for four tiles per workgroup (cols_plan: more tiles than
# CUs, and twice as many), the last tile partly past the rows.
@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("family,n,k", [("dot4", 6396, 768), ("dot4", 12792, 512), ("dot4", 12810, 1280),
                                        ("mfma", 6396, 768), ("mfma", 8182, 2304), ("mfma", 12792, 6144)])
def test_cols_several_tiles_per_workgroup(gpu, orc, tname, family, n, k):
    """Columns in every group count, single launches and two: within the
    bound of the oracle on the first and last rows, and bit-identical to a
    weight that holds these rows alone (one tile per workgroup)."""
    t = TYPES[tname]
    w = orc.random_weight(95, t, n, k)
    rb = w.reshape(n, -1)
    rows = np.r_[0:33, n - 43:n]
    few = np.ascontiguousarray(rb[rows]).reshape(-1)
    gpu.set_kernels(family)
    wg, fg = upload(gpu, t, w, n, k), upload(gpu, t, few, len(rows), k)
    gpu.set_kernels("auto")
    for m in (9, 20, 33, 48, 64, 70):
        if family == "mfma" and (m <= 16 or (m == 64 and tname == "Q8_0" and k < 2560)):
            continue  # (the int8 classes)
        qs, d, s = _q8(orc, 96 + m, m, k)
        xq = q8_1_to_device(gpu, qs, d, s)
        out, part = gpu.alloc(m * n + 8), gpu.alloc(m * len(rows))
        out.fill_(float("nan"))
        gpu.matvec(xq, wg, out, m)
        gpu.matvec(xq, fg, part, m)
        got = gpu.to_host(out)
        assert np.isnan(got[m * n:]).all(), "wrote past the output"
        got = np.ascontiguousarray(got[:m * n].reshape(m, n)[:, rows]).reshape(-1)
        assert np.isfinite(got).all()
        orc.assert_close(f"{tname} {n}x{k} m={m} {family}", orc.matvec_q8_1(t, few, len(rows), k, qs, d, m), got, TOL)
        assert np.array_equal(got.view(np.uint32), gpu.to_host(part, m * len(rows)).view(np.uint32)), f"m={m}"


@pytest.mark.parametrize("family", ["dot4", "mfma"])
@pytest.mark.parametrize("rows", [(4100, 1030, 1100), (6400, 3200, 3300)])
def test_cols_mixed_launch_of_several_tiles(gpu, orc, family, rows):
    """Q4_K and Q6_K in one launch of more tiles than CUs, and than twice as
    many: each output as in its weight's own launch."""
    k, m = 1280, 40
    spec = list(zip((12, 14, 12), rows))
    gpu.set_kernels(family)
    wgs = [upload(gpu, t, orc.random_weight(97 + i, t, n, k), n, k) for i, (t, n) in enumerate(spec)]
    gpu.set_kernels("auto")
    for cols in (9, 17, m, 70):
        x = _q8(orc, 98 + cols, cols, k)
        xq = q8_1_to_device(gpu, *x)
        outs = [gpu.alloc(cols * n) for n in rows]
        gpu.matvec_many(xq, wgs, outs, cols)
        if family == "mfma" and cols <= 16:
            continue  # (the mixed int8 class there)
        for n, wg, out in zip(rows, wgs, outs):
            own = gpu.alloc(cols * n)
            gpu.matvec(xq, wg, own, cols)
            assert torch.equal(own, out), f"{n} rows, {cols} columns"


@pytest.mark.parametrize("tname,n,k,m", [("Q8_0", 6400, 1024, 50), ("Q8_0", 8192, 2304, 64), ("Q4_K", 8192, 4096, 49),
                                         ("Q4_0", 6400, 3584, 64), ("Q4_K", 8208, 4096, 17),
                                         ("Q4_K", 5120, 3584, 100), ("Q8_0", 5120, 2304, 100), ("Q4_K", 9216, 2048, 65),
                                         ("Q4_0", 9216, 4096, 40)])
def test_rows_that_keep_the_16_column_classes(gpu, orc, tname, n, k, m):
    """MFMA layout: more than two tiles per CU of up to 16 super-blocks, and
    past 48 columns more than one of the widths where two launches lose to one
    of the 16-column classes: columns as in a 16-column launch, bit for bit."""
    t = TYPES[tname]
    w = orc.random_weight(92, t, n, k)
    gpu.set_kernels("mfma")
    wg = upload(gpu, t, w, n, k)
    gpu.set_kernels("auto")
    qs, d, s = _q8(orc, 93 + m, m, k)
    out, part = gpu.alloc(m * n), gpu.alloc(16 * n)
    gpu.matvec(q8_1_to_device(gpu, qs, d, s), wg, out, m)
    gpu.matvec(q8_1_to_device(gpu, qs[:16 * k], d[:16 * k // 32], s[:16 * k // 32]), wg, part, 16)
    assert torch.equal(out[:16 * n], part)


@pytest.mark.parametrize("tname,n,k,m", [("Q8_0", 96, 11008, 7), ("Q8_0", 2040, 14336, 9), ("Q6_K", 1024, 11008, 7),
                                         ("Q4_K", 96, 20480, 8), ("Q4_0", 65536, 512, 12), ("Q6_K", 28672, 512, 16),
                                         ("Q8_0", 65600, 1024, 12)])
def test_rows_that_keep_the_dot4_kernels(gpu, orc, tname, n, k, m):
    """Default layout: wide rows on fewer tiles than CUs at 7 to 9 columns, and
    many short rows: columns as in one-column calls, bit for bit."""
    t = TYPES[tname]
    wg = upload(gpu, t, orc.random_weight(94, t, n, k), n, k)
    qs, d, s = _q8(orc, 95 + m, m, k)
    out, one = gpu.alloc(m * n), gpu.alloc(n)
    gpu.matvec(q8_1_to_device(gpu, qs, d, s), wg, out, m)
    for c in (0, m - 1):
        gpu.matvec(q8_1_to_device(gpu, qs[c * k:(c + 1) * k], d[c * k // 32:(c + 1) * k // 32],
                                  s[c * k // 32:(c + 1) * k // 32]), wg, one, 1)
        assert torch.equal(out[c * n:(c + 1) * n], one), f"column {c}"
