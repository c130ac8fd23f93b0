"""Performance cases of the quantized linear-layer path.

Each case is work that a program serving a quantized GGUF model has this
package do, through `rllm_amd.backend.HipBackend`: single projections, the
q/k/v group, the gated FFN and whole transformer layers (attention itself
left out: its output is an input here), for one decoded token, for batches of
tokens and for prompts. Shapes are those of the repository's tests and
benchmark (4096-, 5120- and 8192-wide models), weights are N(0, 0.02) values
quantized to their GGUF type, activations N(0, 1) with a few large channels
as a norm's output has them.

`layout` is the kernel family a weight is uploaded for: "auto" (the default),
"mfma" (what a batching server asks for) or "both".
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rllm_amd.backend import GEMM_MIN_M_DEFAULT, Activation, HipBackend, HostTensor, Q8_1
from rllm_amd.dtype import DType

EPS = 1e-5
TYPES = {"q4_0": DType.Q4_0, "q8_0": DType.Q8_0, "q4_k": DType.Q4_K, "q6_k": DType.Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}


# ---------------------------------------------------------------------------
# The cases.


def _linear(name, weights, cols, m, layout, x):
    return {"name": name, "kind": "linear", "weights": weights, "cols": cols, "m": m, "layout": layout, "input": x}


def _ffn(name, gate, down, cols, ffn, m, layout, x, act="silu"):
    return {"name": name, "kind": "ffn", "gate": gate, "down": down, "cols": cols, "ffn": ffn, "m": m,
            "layout": layout, "input": x, "act": act}


def _layers(name, hidden, kv, ffn, layers, vocab, m, layout):
    return {"name": name, "kind": "layers", "hidden": hidden, "kv": kv, "ffn": ffn, "layers": layers,
            "vocab": vocab, "m": m, "layout": layout}


def listed():
    return [
        # One token's key projection, the smallest call of a decode step: a
        # single launch of 2 MB, all latency.
        _linear("k_proj_1", "q4_k:1024", 4096, 1, "auto", "f32"),
        # Decoding one token: two layers of an 8B-shape model as a decode loop
        # runs them, one captured graph replayed per token.
        _layers("decode_1", 4096, 1024, 14336, 2, 0, 1, "auto"),
        # The vocabulary head for one token, the largest weight of a model.
        _linear("head_1", "q6_k:128256", 4096, 1, "auto", "q8_1"),
        # Two sequences through a Q8_0 gate projection of a 7B-shape model.
        _linear("q8_0_2", "q8_0:11008", 4096, 2, "auto", "f32"),
        # Six sequences decoded together on weights in the default layout.
        _layers("decode_6", 4096, 1024, 14336, 2, 0, 6, "auto"),
        # Sixteen sequences on a batching server's layout, head and logits
        # included: the whole call of a (short) model.
        _layers("decode_16_logits", 4096, 1024, 14336, 2, 128256, 16, "mfma"),
        # The down projection for 32 sequences, both layouts kept.
        _linear("down_32", "q6_k:4096", 14336, 32, "both", "q8_1"),
        # A short prompt of 43 tokens through q/k/v of a 5120-wide model in
        # the default layout.
        _linear("qkv_43", "q4_k:5120,q4_k:5120,q6_k:5120", 5120, 43, "auto", "f32"),
        # A batch of 64 through a Q4_0 projection.
        _linear("q4_0_64", "q4_0:4096", 4096, 64, "mfma", "f32"),
        # A prompt of 100 tokens through a 13B-shape gated FFN.
        _ffn("ffn_100", "q4_k", "q6_k", 5120, 13824, 100, "auto", "f32"),
        # A 512-token prompt through a gate projection.
        _linear("gate_512", "q4_k:14336", 4096, 512, "mfma", "f32"),
        # A 1024-token prompt through a whole 8B-shape layer, the last
        # token's logits at the end.
        _layers("prompt_1024", 4096, 1024, 14336, 1, 128256, 1024, "auto"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: 1 to 1024 tokens, projections
    of 96 to 28672 rows and 512 to 14336 columns (block formats also in widths
    that are no whole super-block), every type and layout."""
    layout = rng.choice(["auto", "auto", "mfma", "both"])
    kind = rng.choice(["linear", "linear", "linear", "ffn", "layers"])
    m = _log_int(rng, 1, 1024)
    if kind == "layers":
        hidden = rng.choice([2048, 4096, 5120])
        ffn = rng.choice({2048: [2048, 5632], 4096: [11008, 14336], 5120: [13824]}[hidden])
        kv = rng.choice([hidden // 4, hidden])
        c = _layers("", hidden, kv, ffn, 1, rng.choice([0, 0, 32000]), m, layout)
    elif kind == "ffn":
        cols = 256 * _log_int(rng, 4, 32)
        ffn = 256 * _log_int(rng, 4, 64)
        gate, down = rng.choice([("q4_k", "q6_k"), ("q4_k", "q4_k"), ("q8_0", "q8_0"), ("q4_0", "q4_0"),
                                 ("q6_k", "q6_k")])
        x = "f32" if m >= GEMM_MIN_M_DEFAULT else rng.choice(["f32", "q8_1"])
        c = _ffn("", gate, down, cols, ffn, m, layout, x, rng.choice(["silu", "gelu"]))
    else:
        t = rng.choice(list(TYPES))
        unit = BLOCK[t][0]
        cols = unit * _log_int(rng, 512 // unit, 14336 // unit)
        rows = _log_int(rng, 96, 28672)
        if rng.random() < 0.6:
            rows = max(32, rows // 32 * 32)
        weights = f"{t}:{rows}"
        if unit == 256 and rng.random() < 0.3:
            kv = max(32, rows // 4)
            weights = f"{t}:{rows},{t}:{kv},{rng.choice([t, 'q6_k'])}:{kv}"
        x = "f32" if m >= GEMM_MIN_M_DEFAULT else rng.choice(["f32", "q8_1"])
        c = _linear("", weights, cols, m, layout, x)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Weights: N(0, 0.02) quantized to GGUF blocks on the GPU.


def _gen(seed, n):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + n) % (1 << 62))
    return g


def _bytes_f16(x):
    return x.to(torch.float16).contiguous().view(torch.uint8)


def _quantize(t, rows, cols, seed, n):
    """GGUF bytes [rows, row_bytes] (uint8, on the GPU) of weight n."""
    g = _gen(seed, n)
    w = torch.randn((rows, cols), generator=g, device="cuda") * 0.02
    e, _ = BLOCK[t]
    nb = cols // e
    if t == "q8_0":
        b = w.view(rows, nb, 32)
        d = (b.abs().amax(-1, keepdim=True) / 127).half()
        q = (b / d.float().clamp_min(1e-12)).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_bytes_f16(d), q], -1).view(rows, -1)
    if t == "q4_0":
        b = w.view(rows, nb, 32)
        big = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        d = (big / -8).half()
        q = (b / d.float() + 8).round().clamp(0, 15).to(torch.uint8)
        return torch.cat([_bytes_f16(d), q[..., :16] | (q[..., 16:] << 4)], -1).view(rows, -1)
    if t == "q4_k":
        b = w.view(rows, nb, 8, 32)
        lo = (-b.amin(-1)).clamp_min(0)
        sc = (b.amax(-1) + lo) / 15
        d = (sc.amax(-1, keepdim=True) / 63).half()
        dm = (lo.amax(-1, keepdim=True) / 63).half()
        isc = (sc / d.float()).round().clamp(1, 63)
        imn = (lo / dm.float()).round().clamp(0, 63)
        q = ((b + (dm.float() * imn)[..., None]) / (d.float() * isc)[..., None]).round().clamp(0, 15).to(torch.uint8)
        s, m = isc.to(torch.uint8), imn.to(torch.uint8)
        packed = torch.cat([s[..., :4] | ((s[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                            (s[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
        qs = q[..., 0::2, :] | (q[..., 1::2, :] << 4)
        return torch.cat([_bytes_f16(d), _bytes_f16(dm), packed, qs.flatten(-2)], -1).view(rows, -1)
    b = w.view(rows, nb, 16, 16)  # q6_k: signed sub-block scales
    sign = torch.randint(0, 2, (rows, nb, 16), generator=g, device="cuda") * 2 - 1
    sc = b.abs().amax(-1) / 31
    d = (sc.amax(-1, keepdim=True) / 127).half()
    isc = (sc / d.float()).round().clamp(1, 127) * sign
    q = ((b / (d.float() * isc)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(rows, nb, 2, 4, 32)
    ql = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -1)
    qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
    return torch.cat([ql.flatten(-2), qh.flatten(-2), isc.to(torch.int8).view(torch.uint8), _bytes_f16(d)], -1).view(rows, -1)


def _dequantize(t, raw, cols):
    """float64 [rows, cols] of GGUF bytes [rows, row_bytes]."""
    rows = raw.shape[0]
    e, nbytes = BLOCK[t]
    b = raw.view(rows, cols // e, nbytes)

    def f16(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()

    if t == "q8_0":
        return (f16(0) * b[..., 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    if t == "q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        return (f16(0) * q).view(rows, cols)
    if t == "q4_k":
        p = b[..., 4:16]
        sc = torch.cat([p[..., :4] & 63, (p[..., 8:] & 15) | ((p[..., :4] >> 6) << 4)], -1).double()
        mn = torch.cat([p[..., 4:8] & 63, (p[..., 8:] >> 4) | ((p[..., 4:8] >> 6) << 4)], -1).double()
        qs = b[..., 16:].reshape(rows, -1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], -2).reshape(rows, -1, 8, 32).double()
        return ((f16(0) * sc)[..., None] * q - (f16(2) * mn)[..., None]).view(rows, cols)
    ql, qh = b[..., :128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 1, 32)
    hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
    q = (torch.cat([ql & 15, ql >> 4], -2) | (hi << 4)).reshape(rows, -1, 16, 16).double() - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return ((f16(208) * sc)[..., None] * q).view(rows, cols)


# ---------------------------------------------------------------------------
# Activations.


def _act(seed, n, m, k):
    """f32 [m, k]: N(0, 1), every 64th channel or so several times larger."""
    g = _gen(seed, 1000 + n)
    x = torch.randn((m, k), generator=g, device="cuda")
    big = torch.rand((k,), generator=g, device="cuda") < 1 / 64
    return torch.where(big, x * 6, x).contiguous()


def _norm_weight(seed, n, k):
    return 1 + 0.1 * torch.randn((k,), generator=_gen(seed, 2000 + n), device="cuda")


def _q8_codes(x):
    """Q8_1 of x [m, k] as its definition gives it: int8 codes [m, k/32, 32]
    and the f16 scale, with 32-bit IEEE divisions (on the host)."""
    x = x.detach().to("cpu", torch.float32)
    b = x.view(x.shape[0], -1, 32).numpy()
    d = np.abs(b).max(-1, keepdims=True) / np.float32(127)
    with np.errstate(divide="ignore", invalid="ignore"):
        q = np.where(d > 0, np.rint(b / d), 0)
    return q.astype(np.int8), d.astype(np.float16)


def _q8_values(x):
    """The float64 values Q8_1 of x stands for."""
    q, d = _q8_codes(x)
    v = q.astype(np.float64) * d.astype(np.float64)
    return torch.from_numpy(v).view(x.shape).to("cuda")


def _q8_tensor(be, x, m, k):
    """x as its producer left it, in Q8_1."""
    return be.quantize_q8_1(x, m, k)


# ---------------------------------------------------------------------------
# States.

_BE = None


def _backend():
    global _BE
    if _BE is None:
        _BE = HipBackend(0)
    _BE.set_stream(torch.cuda.current_stream())
    return _BE


def _upload(be, layout, t, rows, cols, seed, n):
    be.set_kernels(layout)
    raw = _quantize(t, rows, cols, seed, n).cpu().numpy()
    return be.upload(HostTensor(f"w{n}", TYPES[t], (rows, cols), raw))


def _parts(case):
    return [(t, int(r)) for t, r in (p.split(":") for p in case["weights"].split(","))]


def _empty(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def _layer_shapes(case):
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [("q4_k", h, h), ("q4_k", kv, h), ("q6_k", kv, h), ("q4_k", h, h), ("q4_k", f, h), ("q4_k", f, h), ("q6_k", h, f)]


class _State:
    pass


def prepare(case, seed):
    be = _backend()
    s = _State()
    s.case, s.be, s.graph = case, be, None
    m, layout = case["m"], case["layout"]
    if case["kind"] == "linear":
        k = case["cols"]
        s.ws = [_upload(be, layout, t, r, k, seed, i) for i, (t, r) in enumerate(_parts(case))]
        s.outs = [_empty(m, w.rows) for w in s.ws]
        s.x = _act(seed, 0, m, k)
        be.reserve(m * k)
        if case["input"] == "q8_1":
            s.xq = _q8_tensor(be, s.x, m, k)
    elif case["kind"] == "ffn":
        k, f = case["cols"], case["ffn"]
        s.ws = [_upload(be, layout, t, r, c, seed, i)
                for i, (t, r, c) in enumerate([(case["gate"], f, k), (case["gate"], f, k), (case["down"], k, f)])]
        s.x = _act(seed, 0, m, k)
        s.out, s.h, s.u = _empty(m, k), _empty(m, f), _empty(m, f)
        be.reserve(m * max(k, f))
        if case["input"] == "q8_1":
            s.xq = _q8_tensor(be, s.x, m, k)
    else:
        _prepare_layers(s, seed)
    torch.cuda.synchronize()
    return s


def _prepare_layers(s, seed):
    case, be = s.case, s.be
    m, h, kv, f = case["m"], case["hidden"], case["kv"], case["ffn"]
    s.int8 = m < GEMM_MIN_M_DEFAULT
    s.x0 = _act(seed, 0, m, h)
    s.x, s.hn, s.fo, s.gate, s.up = _empty(m, h), _empty(m, h), _empty(m, h), _empty(m, f), _empty(m, f)
    s.hq = Q8_1.empty(m * h, be.device) if s.int8 else None
    be.reserve(m * f)
    s.layers = []
    for i in range(case["layers"]):
        layer = _State()
        layer.ws = [_upload(be, case["layout"], t, r, c, seed, 10 * i + j)
                    for j, (t, r, c) in enumerate(_layer_shapes(case))]
        layer.n1, layer.n2 = _norm_weight(seed, 2 * i, h), _norm_weight(seed, 2 * i + 1, h)
        layer.att = _act(seed, 10 + i, m, h)
        layer.attq = _q8_tensor(be, layer.att, m, h) if s.int8 else None
        layer.qkv = [_empty(m, h), _empty(m, kv), _empty(m, kv)]
        layer.o, layer.fo = _empty(m, h), _empty(m, h)
        s.layers.append(layer)
    s.nf = _norm_weight(seed, 99, h)
    s.head = _upload(be, case["layout"], "q6_k", case["vocab"], h, seed, 999) if case["vocab"] else None
    s.logits = _empty(m if s.int8 else 1, case["vocab"]) if case["vocab"] else None
    if not s.int8:
        return
    # A decode loop captures its step once and replays it for every token.
    home = torch.cuda.current_stream()
    _run_layers(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        be.set_stream(torch.cuda.current_stream())
        _run_layers(s)
    be.set_stream(home)
    s.graph = graph


def _run_layers(s):
    case, be = s.case, s.be
    m, h = case["m"], case["hidden"]
    s.x.copy_(s.x0)
    prev = None
    for layer in s.layers:
        q, k, v, o, gate, up, down = layer.ws
        if prev is None:
            be.rms_norm(s.x, layer.n1, s.hn, m, EPS, s.hq)
        else:
            be.add_rms_norm(s.x, prev, layer.n1, s.hn, m, h, EPS, s.hq)
        if s.int8:
            be.matvec_many(s.hq, [q, k, v], layer.qkv, m)
            be.matvec(layer.attq, o, layer.o, m)
        else:
            be.matmul_many(s.hn, [q, k, v], layer.qkv, m)
            be.matmul(layer.att, o, layer.o, m)
        be.add_rms_norm(s.x, layer.o, layer.n2, s.hn, m, h, EPS, s.hq)
        if s.int8:
            be.gated_ffn_q8_1(s.hq, gate, up, down, Activation.SILU, layer.fo, s.gate, s.up, m)
        else:
            be.gated_ffn(s.hn, gate, up, down, Activation.SILU, layer.fo, s.gate, s.up, m)
        prev = layer.fo
    be.add_rms_norm(s.x, prev, s.nf, s.hn, m, h, EPS, s.hq)
    if s.head is not None:
        if s.int8:
            be.matvec(s.hq, s.head, s.logits, m)
        else:
            be.matmul(s.hn[m - 1], s.head, s.logits, 1)


def run(s):
    case, be = s.case, s.be
    m = case["m"]
    if case["kind"] == "linear":
        if case["input"] == "q8_1":
            if len(s.ws) == 1:
                be.matvec(s.xq, s.ws[0], s.outs[0], m)
            else:
                be.matvec_many(s.xq, s.ws, s.outs, m)
        elif len(s.ws) == 1:
            be.matmul(s.x, s.ws[0], s.outs[0], m)
        else:
            be.matmul_many(s.x, s.ws, s.outs, m)
        return s.outs
    if case["kind"] == "ffn":
        act = Activation.SILU if case["act"] == "silu" else Activation.GELU_TANH
        if case["input"] == "q8_1":
            be.gated_ffn_q8_1(s.xq, *s.ws, act, s.out, s.h, s.u, m)
        else:
            be.gated_ffn(s.x, *s.ws, act, s.out, s.h, s.u, m)
        return [s.h, s.out]
    if s.graph is not None:
        s.graph.replay()
    else:
        _run_layers(s)
    outs = [t for layer in s.layers for t in (*layer.qkv, layer.o, layer.fo)] + [s.x]
    return outs + ([s.logits] if s.logits is not None else [])


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what it should return.


def _weight_bytes(t, rows, cols):
    e, b = BLOCK[t]
    return rows * cols // e * b


def work(case):
    m = case["m"]
    if case["kind"] == "linear":
        k = case["cols"]
        w = [(t, r, k) for t, r in _parts(case)]
        act = m * k * 4 if case["input"] == "f32" else m * k // 32 * 36
        act += 4 * m * sum(r for _, r, _ in w)
        rows_m = [m] * len(w)
    elif case["kind"] == "ffn":
        k, f = case["cols"], case["ffn"]
        w = [(case["gate"], f, k), (case["gate"], f, k), (case["down"], k, f)]
        act = (m * k * 4 if case["input"] == "f32" else m * k // 32 * 36) + 4 * m * (f + k)
        rows_m = [m] * 3
    else:
        h, kv = case["hidden"], case["kv"]
        w = _layer_shapes(case) * case["layers"]
        rows_m = [m] * len(w)
        # In: the embedding, the attention outputs and the norm weights; out:
        # q, k, v, o, the FFN's output per layer, x and the logits.
        int8 = m < GEMM_MIN_M_DEFAULT
        act = 4 * m * h * 2 + 4 * h
        act += case["layers"] * (8 * h + (m * h // 32 * 36 if int8 else 4 * m * h) + 4 * m * (3 * h + 2 * kv))
        if case["vocab"]:
            w = w + [("q6_k", case["vocab"], h)]
            rows_m.append(m if int8 else 1)
            act += 4 * rows_m[-1] * case["vocab"]
    return {"bytes": sum(_weight_bytes(*x) for x in w) + act,
            "flops": sum(2 * r * c * mm for (_, r, c), mm in zip(w, rows_m))}


def tolerance(case):
    """Measured against `exact`, about four times what was seen.

    Below GEMM_MIN_M_DEFAULT columns the block dots are whole numbers and
    their sums 32-bit (1.9e-7). A gated FFN rounds its product to Q8_1 on the
    way, a layer its norms' outputs too: another order of the sums before them
    moves a few codes by one step (1/127 of a block's largest value), which
    the next layers pass on (4e-3 to 7e-3 after two layers). From there on weights and
    activations may be held in f16, 2^-11 each (2.9e-4 for a product, 5e-4
    after an FFN); a prompt's last token goes to the head in Q8_1 (3e-3).
    """
    int8 = case["m"] < GEMM_MIN_M_DEFAULT or case.get("input") == "q8_1"
    if case["kind"] == "linear":
        return {"rel": 1e-6} if int8 else {"rel": 1.2e-3}
    if case["kind"] == "ffn":
        return {"rel": 1e-3} if int8 else {"rel": 2e-3}
    return {"rel": 2.5e-2} if int8 else {"rel": 1.2e-2}


def _apply(act, g, u):
    if act == "silu":
        return g / (1 + torch.exp(-g)) * u
    return 0.5 * g * (1 + torch.tanh(0.7978845608 * (g + 0.044715 * g ** 3))) * u


def exact(case, seed):
    m = case["m"]
    if case["kind"] == "linear":
        k = case["cols"]
        int8 = m < GEMM_MIN_M_DEFAULT or case["input"] == "q8_1"
        x = _act(seed, 0, m, k)
        xv = _q8_values(x) if int8 else x.double()
        outs = []
        for i, (t, r) in enumerate(_parts(case)):
            outs.append(_product(xv, t, r, k, seed, i))
        return outs
    if case["kind"] == "ffn":
        k, f = case["cols"], case["ffn"]
        int8 = m < GEMM_MIN_M_DEFAULT or case["input"] == "q8_1"
        x = _act(seed, 0, m, k)
        xv = _q8_values(x) if int8 else x.double()
        g = _product(xv, case["gate"], f, k, seed, 0)
        h = _apply(case["act"], g, _product(xv, case["gate"], f, k, seed, 1))
        return [h, _product(_q8_values(h) if int8 else h, case["down"], k, f, seed, 2)]
    h, f = case["hidden"], case["ffn"]
    int8 = m < GEMM_MIN_M_DEFAULT
    values = _q8_values if int8 else (lambda v: v.double())

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()

    x = _act(seed, 0, m, h).double()
    outs = []
    for i in range(case["layers"]):
        def mul(v, j):
            t, r, c = _layer_shapes(case)[j]
            return _product(v, t, r, c, seed, 10 * i + j)

        hv = values(norm(x, _norm_weight(seed, 2 * i, h)))
        outs += [mul(hv, 0), mul(hv, 1), mul(hv, 2)]
        outs.append(mul(values(_act(seed, 10 + i, m, h)), 3))
        x = x + outs[-1]
        hv = values(norm(x, _norm_weight(seed, 2 * i + 1, h)))
        outs.append(mul(values(_apply("silu", mul(hv, 4), mul(hv, 5))), 6))
        x = x + outs[-1]
    outs.append(x)
    if case["vocab"]:
        hn = norm(x, _norm_weight(seed, 99, h))
        # For a prompt only its last token's logits, one column: the int8 path.
        hv = values(hn) if int8 else _q8_values(hn[m - 1:])
        outs.append(_product(hv, "q6_k", case["vocab"], h, seed, 999))
    return outs


def _product(xv, t, rows, cols, seed, n):
    """float64 [m, rows] = xv . dequantized(weight n)^T, a slab of rows at a time."""
    raw = _quantize(t, rows, cols, seed, n)
    out = torch.empty((xv.shape[0], rows), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // cols)
    for lo in range(0, rows, step):
        w = _dequantize(t, raw[lo:lo + step].contiguous(), cols)
        out[:, lo:lo + step] = xv @ w.t().contiguous()
    return out
