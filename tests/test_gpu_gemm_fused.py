"""The f16 GEMM route's kernels that dequantize in registers (rq_gemm_*), at
the edges of their row blocks, column groups and super-blocks: against the
exact product of the f16 values, both layouts bit-identical, and beside
weights that stay with the vendor GEMM."""
import numpy as np
import pytest
import torch

from gpu_util import make_weight, upload
from rllm_amd.backend import HipBackend
from rllm_amd.errors import BackendError, ShapeError

pytestmark = pytest.mark.gpu

TYPES = {"Q4_0": 2, "Q8_0": 8, "Q4_K": 12, "Q6_K": 14}

# Against f64 over both operands rounded to f16, the very values the kernels
# multiply (test_gemm_fused_weights_are_the_copys): what is left are the f32
# sums, within 1e-5 of the largest output as in the matvecs; five times that.
TOL = 5e-5


def _exact(orc, t, w, n, k, x, m):
    f16 = lambda v: v.astype(np.float16).astype(np.float64)
    return (f16(x.reshape(m, k)) @ f16(orc.dequantize(t, w, n, k).reshape(n, k)).T).reshape(-1)


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("n,k", [(1, 256), (17, 2048), (32, 2304), (70, 4096), (300, 14336), (33, 32), (50, 2080)])
@pytest.mark.parametrize("m", [65, 96, 97, 128, 129, 192, 193, 256, 500])
def test_gemm_fused(gpu, orc, tname, n, k, m):
    t = TYPES[tname]
    if t in (12, 14) and k % 256:
        pytest.skip("K-quants need k % 256 == 0")
    w = make_weight(orc, t, n, k, 60 + n, "normal")
    x = orc.normal(61 + k + m, m * k, 0.0, 1.0)
    xg = gpu.from_host(x)
    want, got = _exact(orc, t, w, n, k, x, m), {}
    for fam in ("dot4", "mfma"):
        gpu.set_kernels(fam)
        wg = upload(gpu, t, w, n, k)
        gpu.set_kernels("auto")
        out = gpu.alloc(m * n + 8)
        out.fill_(float("nan"))
        gpu.matmul(xg, wg, out, m)
        got[fam] = gpu.to_host(out)
        assert np.isnan(got[fam][m * n:]).all(), "wrote past the output"
        orc.assert_close(f"{tname} {n}x{k} m={m} {fam}", want, got[fam][:m * n], TOL)
    if m <= 256 or k < 8192:  # (past them: the vendor GEMM on the copy)
        assert np.array_equal(got["dot4"][:m * n].view(np.uint32), got["mfma"][:m * n].view(np.uint32))


@pytest.mark.parametrize("m", [65, 100])
@pytest.mark.parametrize("k", [4096, 14336])
def test_gemm_fused_beside_kept_copies(gpu, orc, k, m):
    """matmul_many over weights on both sides of the rule (a weight with a kept
    copy goes to the vendor GEMM, at k = 14336 in slices of k): each as in its
    own call, and replayed from a graph after reserve_f16."""
    t, rows = 12, (200, 300, 72)
    ws = [make_weight(orc, t, n, k, 70 + n, "normal") for n in rows]
    wgs = [upload(gpu, t, w, n, k) for w, n in zip(ws, rows)]
    gpu.keep_f16(wgs[1])
    x = orc.normal(71 + m, m * k, 0.0, 1.0)
    gpu.reserve_f16(max(rows) * k, m * k, m * max(rows))
    xg = gpu.from_host(x)
    own = [gpu.alloc(m * n) for n in rows]
    for wg, out in zip(wgs, own):
        gpu.matmul(xg, wg, out, m)
    for w, n, out in zip(ws, rows, own):
        orc.assert_close(f"{n}x{k} m={m}", _exact(orc, t, w, n, k, x, m), gpu.to_host(out), TOL)
    outs = [gpu.alloc(m * n) for n in rows]
    gpu.matmul_many(xg, wgs, outs, m)
    gpu.synchronize()
    for a, b in zip(own, outs):
        assert torch.equal(a, b)
    graph, stream, main = torch.cuda.CUDAGraph(), torch.cuda.Stream(gpu.device), gpu.stream
    torch.cuda.synchronize()
    gpu.set_stream(stream)
    try:
        with torch.cuda.graph(graph, stream=stream):
            gpu.matmul_many(xg, wgs, outs, m)
    finally:
        gpu.set_stream(main)
    for _ in range(3):
        for b in outs:
            b.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(own, outs):
            assert torch.equal(a, b)


def _one_hot(gpu, k, m, first):
    """m columns, column j one-hot at element first + j (zeros past k)."""
    x = torch.zeros((m, k), dtype=torch.float32, device=gpu.device)
    for j in range(min(m, k - first)):
        x[j, first + j] = 1.0
    return x


@pytest.mark.parametrize("family", ["dot4", "mfma"])
@pytest.mark.parametrize("m", [96, 128])
@pytest.mark.parametrize("tname", list(TYPES))
def test_gemm_fused_weights_are_the_copys(gpu, orc, tname, family, m):
    """The f16 weights made in registers are those of the dequantized copy
    (rq_dequant_f16), bit for bit: a one-hot column's product is one weight.
    Q4_K's super-blocks hold f16 ties: d sc q has 12 significant bits, the last
    one set, and dmin m is less than half a unit of it in f32, so that the f32
    difference is the tie and rounds to even, where rounded once from the exact
    difference it would go down."""
    t, n, k = TYPES[tname], 64, 256
    w = make_weight(orc, t, n, k, 80, "random")
    if t == 12:
        b = w.reshape(n, 144)
        odd = np.random.default_rng(81).integers(512, 1024, n) * 2 + 1  # 11 bits, odd
        b[:, 0:2] = (odd.astype(np.float32) * 2.0 ** -9).astype(np.float16).view(np.uint8).reshape(n, 2)  # d in 2..4
        b[:, 2:4] = np.full((n, 1), 2.0 ** -24, np.float16).view(np.uint8)  # dmin: the least f16
        b[:, 4:16] = np.array([1] * 8 + [0x11] * 4, np.uint8)  # every scale and min 1
    gpu.set_kernels(family)
    wg = upload(gpu, t, w, n, k)
    gpu.set_kernels("auto")
    want = gpu.dequant_f16(wg).reshape(n, k).float()
    got = torch.empty((n, k), device=gpu.device)
    for first in range(0, k, m):
        out = gpu.alloc(m * n)
        gpu.matmul(_one_hot(gpu, k, m, first).reshape(-1), wg, out, m)
        cols = min(m, k - first)
        got[:, first:first + cols] = out[:m * n].reshape(m, n)[:cols].t()
    bad = int((got != want).sum())
    assert bad == 0, f"{bad} of {n * k} weights differ"


@pytest.mark.filterwarnings("ignore:The CUDA Graph is empty")
def test_gemm_fused_takes_no_copy_scratch(gpu, orc):
    """A call whose weights are all dequantized in registers needs x's scratch
    alone: no f16 copy of a weight (32 MB here) and no vendor workspace (64
    MB), and it can be captured with nothing reserved for a weight."""
    t, n, k, m = 12, 4096, 4096, 100
    w = orc.random_weight(82, t, n, k)
    fresh = HipBackend(gpu.device.index or 0)
    try:
        wg = upload(fresh, t, w, n, k)
        x = fresh.from_host(orc.normal(83, m * k, 0.0, 1.0))
        out = fresh.alloc(m * n)
        graph, stream, main = torch.cuda.CUDAGraph(), torch.cuda.Stream(fresh.device), fresh.stream

        def capture():
            torch.cuda.synchronize()
            fresh.set_stream(stream)
            try:
                with torch.cuda.graph(graph, stream=stream):
                    fresh.matmul(x, wg, out, m)
            finally:
                fresh.set_stream(main)

        with pytest.raises(ShapeError, match="rq_reserve_f16"):
            capture()
        torch.cuda.synchronize()
        free0, _ = torch.cuda.mem_get_info(fresh.device)
        fresh.matmul(x, wg, out, m)
        fresh.synchronize()
        free1, _ = torch.cuda.mem_get_info(fresh.device)
        assert free0 - free1 < 16 << 20, f"the call took {free0 - free1} bytes"
        want = out.clone()
        graph = torch.cuda.CUDAGraph()
        capture()
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
        del graph
    finally:
        fresh.synchronize()
        fresh.close()


def test_reserve_f16_refuses_more_than_there_is(gpu):
    """Reservations past any memory fail in the allocator, also where the
    padded size of x's scratch would not fit 64 bits."""
    fresh = HipBackend(gpu.device.index or 0)
    try:
        for values in (1 << 50, (1 << 63) // 80 + 1, 1 << 60):
            with pytest.raises(BackendError):
                fresh.reserve_f16(0, values, 0)
            torch.zeros(1, device=fresh.device).add_(1)  # the failure is the library's alone
            torch.cuda.synchronize()
        fresh.reserve_f16(0, 4096, 0)
    finally:
        fresh.close()


@pytest.mark.parametrize("tname", ["Q4_K", "Q8_0"])
@pytest.mark.parametrize("n,k,m", [(96, 14336, 65), (1024, 14336, 128), (2048, 14336, 112), (1024, 8192, 200),
                                   (28672, 512, 256), (14336, 512, 200), (96, 6144, 400)])
def test_gemm_fused_leaves_what_the_copy_does_faster(gpu, orc, tname, n, k, m):
    """Few rows of many super-blocks, and many rows of few: such products stay
    with the copy and the vendor GEMM, and so have the bits of a kept copy."""
    t = TYPES[tname]
    wg = upload(gpu, t, orc.random_weight(84, t, n, k), n, k)
    x = gpu.from_host(orc.normal(85, m * k, 0.0, 1.0))
    got, want = gpu.alloc(m * n), gpu.alloc(m * n)
    gpu.matmul(x, wg, got, m)
    gpu.keep_f16(wg)
    gpu.matmul(x, wg, want, m)
    assert torch.equal(got, want)
    wg.free()
