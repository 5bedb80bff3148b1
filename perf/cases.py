"""Timed cases of the MoE expert layer: routing from router logits,
segmentation, grouped gate/up + clamped SwiGLU, down, weighted combine.

A case is one or more layers of a model, each called through
``layer.moe_forward`` with the router logits (the call the quant-method hook
makes).  Decode batches (T <= 256 tokens) are captured into a HIP graph when
the model is loaded and replayed per step, as a serving engine runs them;
prefill chunks are called eagerly.  A case's ``layers`` are distinct layers
of one model, each with its own weights and its own rows.

Shapes: the DeepSeek-V3 MoE layer (256 + 1 experts, grouped sigmoid top-8
with a selection bias), the Qwen3-Next one (512 + 1, softmax top-10, SwiGLU
limit 7), a 128-expert layer (softmax top-8) and a tiny Mixtral (8 experts,
top-2).
"""
from __future__ import annotations

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "vllm-xtu-moe_amd"))

from xtu_moe_amd import formats as F  # noqa: E402
from xtu_moe_amd.layer import ExpertWeights, moe_forward  # noqa: E402

DEV = "cuda"
GRAPH_MAX_TOKENS = 256   # decode batches up to this size run as a captured graph
STD = 0.02               # standard deviation of the weights
CHUNK = 16               # experts quantised at a time

SHAPES = {
    "ds": dict(E=256, shared=1, H=7168, I=2048, K=8, grouped=True, limit=0.0),
    "qwen": dict(E=512, shared=1, H=2048, I=512, K=10, grouped=False, limit=7.0),
    "e128": dict(E=128, shared=0, H=2048, I=768, K=8, grouped=False, limit=0.0),
    "tiny": dict(E=8, shared=0, H=1024, I=2048, K=2, grouped=False, limit=0.0),
}
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _case(name, shape, fmt, T, layers=1, int8=False):
    c = dict(shape=shape, fmt=fmt, T=T, layers=layers, int8=int8)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user's decode step: latency, four layers of the step's graph
        _case("qwen-mxfp4-t1", "qwen", "mxfp4", 1, layers=4),
        # a few users (or a draft's tokens) at decode, 4-bit with e4m3 scales
        _case("qwen-nvfp4-t4", "qwen", "nvfp4", 4, layers=4),
        # the large model's decode step at two users
        _case("ds-mxfp4-t2", "ds", "mxfp4", 2, layers=2),
        # its decode at a full small batch
        _case("ds-mxfp4-t16", "ds", "mxfp4", 16),
        # FP8 checkpoint served to a batch of 64 sequences
        _case("e128-fp8-t64", "e128", "fp8", 64),
        # a ragged decode batch over many small experts (most hold one or two rows)
        _case("qwen-nvfp4-t93", "qwen", "nvfp4", 93),
        # unquantised experts, a batch of 128
        _case("tiny-bf16-t128", "tiny", "bf16", 128),
        # decode plus a short prompt in one step: every expert active, few rows each
        _case("ds-mxfp4-t209", "ds", "mxfp4", 209),
        # a prompt of a thousand tokens with int8 activations (the option's own range)
        _case("qwen-int8-t1000", "qwen", "mxfp4", 1000, int8=True),
        # chunked prefill of the FP8 checkpoint at its native block scales
        _case("ds-fp8-t2048", "ds", "fp8", 2048),
        # long prefill over small experts
        _case("qwen-nvfp4-t4096", "qwen", "nvfp4", 4096),
        # long prefill of the large model
        _case("ds-mxfp4-t8192", "ds", "mxfp4", 8192),
    ]


def draw(rng):
    shape, fmt, lo, hi, int8 = rng.choice([
        ("ds", "mxfp4", 1, 8192, False), ("ds", "fp8", 1, 2048, False),
        ("qwen", "mxfp4", 1, 8192, False), ("qwen", "nvfp4", 1, 8192, False),
        ("qwen", "mxfp4", 160, 8192, True), ("e128", "fp8", 1, 8192, False),
        ("e128", "bf16", 1, 4096, False), ("tiny", "bf16", 1, 4096, False),
    ])
    T = min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))
    return _case(None, shape, fmt, T, layers=(2 if shape == "ds" else 4) if T <= 4 else 1,
                 int8=int8)


# ------------------------------------------------------------------ inputs
def _e2m1(v):
    """Nearest e2m1 codes of v (values past 6 saturate)."""
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=v.device)
    return torch.bucketize(v.abs(), mids).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)


def _pow2_floor(v):
    return torch.exp2(torch.floor(torch.log2(v)))


def _quantize(fmt, w):
    """[n, N, K] -> checkpoint planes (codes, scales, second-level scale)."""
    n, N, K = w.shape
    if fmt == "bf16":
        return w.to(torch.bfloat16), None, None
    if fmt == "fp8":
        b = w.view(n, N // 128, 128, K // 128, 128)
        s = b.abs().amax((2, 4)) / 448.0
        q = (b / s[:, :, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
        return q.view(torch.uint8).view(n, N, K), s, None
    g = 32 if fmt == "mxfp4" else 16
    b = w.view(n, N, K // g, g)
    amax = b.abs().amax(-1)
    if fmt == "mxfp4":
        s = _pow2_floor(amax.clamp_min(2.0 ** -100)) / 4
        scales, gs = torch.round(torch.log2(s) + 127).to(torch.uint8), None
    else:
        gs = amax.amax((1, 2)) / (448.0 * 6.0)
        s8 = (amax / 6.0 / gs[:, None, None]).clamp(2.0 ** -6, 448.0).to(torch.float8_e4m3fn)
        s, scales = s8.float() * gs[:, None, None], s8.view(torch.uint8)
    c = _e2m1(b / s[..., None]).view(n, N, K)
    return c[..., 0::2] | (c[..., 1::2] << 4), scales, gs


def _planes(case, gen):
    """One layer's checkpoint planes, in chunks of experts."""
    s = SHAPES[case["shape"]]
    n, H, I, fmt = s["E"] + s["shared"], s["H"], s["I"], case["fmt"]
    for e0 in range(0, n, CHUNK):
        m = min(CHUNK, n - e0)
        w = torch.empty((m, 2 * I, H), device=DEV).normal_(0, STD, generator=gen)
        if fmt == "nvfp4":   # gate and up each with its own second-level scale
            cg, sg, gg = _quantize(fmt, w[:, :I].contiguous())
            cu, su, gu = _quantize(fmt, w[:, I:].contiguous())
            p13 = (torch.cat([cg, cu], 1), torch.cat([sg, su], 1), torch.stack([gg, gu], 1))
        else:
            p13 = _quantize(fmt, w)
        w = torch.empty((m, H, I), device=DEV).normal_(0, STD, generator=gen)
        yield p13 + _quantize(fmt, w)


def _tokens(case, gen):
    """One layer's rows, router logits and selection bias."""
    s = SHAPES[case["shape"]]
    x = torch.empty((case["T"], s["H"]), device=DEV).normal_(0, 1, generator=gen)
    logits = torch.empty((case["T"], s["E"]), device=DEV).normal_(0, 1, generator=gen)
    bias = torch.empty(s["E"], device=DEV).normal_(0, 0.02, generator=gen) if s["grouped"] else None
    return x.to(torch.bfloat16), logits, bias


def _generator(seed, layer):
    return torch.Generator(device=DEV).manual_seed(seed * 64 + layer)


def prepare(case, seed):
    s = SHAPES[case["shape"]]
    fmt = F.fmt_of(case["fmt"])
    layers = []
    for l in range(case["layers"]):
        gen = _generator(seed, l)
        x, logits, bias = _tokens(case, gen)
        parts = list(zip(*_planes(case, gen)))
        cat = [None if p[0] is None else torch.cat(p) for p in parts]
        del parts
        W = ExpertWeights.from_dense(fmt, cat[0], cat[1], cat[3], cat[4], cat[2], cat[5],
                                     n_shared=s["shared"])
        if case["int8"]:
            W.int8_planes()
        router = dict(logits=logits, scoring="softmax")
        if s["grouped"]:
            router.update(scoring="sigmoid", bias=bias, n_group=8, topk_group=4,
                          routed_scaling_factor=2.5)
        T = case["T"]
        layers.append(dict(
            x=x, W=W, router=router, limit=s["limit"], int8=case["int8"],
            ids=torch.empty((T, s["K"]), dtype=torch.int32, device=DEV),
            weights=torch.empty((T, s["K"]), device=DEV),
            out=torch.empty((T, s["H"]), dtype=torch.bfloat16, device=DEV)))
    state = dict(layers=layers, graph=None)
    if case["T"] <= GRAPH_MAX_TOKENS:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(layers)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            _step(layers)
        state["graph"] = graph
    return state


def _step(layers):
    for l in layers:
        moe_forward(l["x"], l["ids"], l["weights"], l["W"], swiglu_limit=l["limit"], out=l["out"],
                    int8=l["int8"], router=l["router"])


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        _step(state["layers"])
    return [{"out": l["out"], "ids": l["ids"], "weights": l["weights"]} for l in state["layers"]]


# ------------------------------------------------------------------- work
def work(case):
    """Every active expert's planes once (the expected number of distinct
    experts of T uniform choices of K), rows and logits in, rows out."""
    s = SHAPES[case["shape"]]
    T, E, H, I, K = case["T"], s["E"], s["H"], s["I"], s["K"]
    n = E * (1.0 - (1.0 - K / E) ** T) + s["shared"]
    bits = {"mxfp4": 4 + 8 / 32, "nvfp4": 4 + 8 / 16, "fp8": 8 + 32 / 16384, "bf16": 16}
    per = 3 * H * I * bits[case["fmt"]] / 8
    nbytes = n * per + T * (2 * H + 4 * E) + T * (2 * H + 8 * K)
    flops = 2.0 * 3 * H * I * T * (K + s["shared"])
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    # bf16 rows out, the SwiGLU rows rounded to bf16 between the two products
    return {"rel": 1e-2, "max": 5e-2, "differ": 1e-4}


# ------------------------------------------------------------------ exact
def _dequantize(fmt, q, s, gs):
    """Checkpoint planes of some experts as float64 [n, N, K]."""
    if fmt == "bf16":
        return q.double()
    n, N = q.shape[0], q.shape[1]
    if fmt == "fp8":
        v = q.view(torch.float8_e4m3fn).double().view(n, N // 128, 128, -1, 128)
        return (v * s.double()[:, :, None, :, None]).view(n, N, -1)
    lut = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=q.device)
    v = torch.stack([lut[(q & 15).long()], lut[(q >> 4).long()]], -1).view(n, N, -1)
    if fmt == "mxfp4":
        sc = torch.exp2(s.double() - 127)
    else:
        sc = s.view(torch.float8_e4m3fn).double()
        sc = (sc.view(n, gs.shape[1], -1) * gs.double()[:, :, None]).view(n, N, -1) \
            if gs.dim() == 2 else sc * gs.double()[:, None, None]
    return (v.view(n, N, sc.shape[2], -1) * sc[..., None]).view(n, N, -1)


def _int8_rows(a):
    """Rows rounded to int8 steps of a power of two per row, as values."""
    m = a.abs().amax(1, keepdim=True).clamp_min(2.0 ** -100)
    e = torch.floor(torch.log2(m))
    e = e - 6 + (m / torch.exp2(e) > 1 + 8257536 / 8388608)
    return torch.round(a * torch.exp2(-e)).clamp(-127, 127) * torch.exp2(e)


def _route(case, logits, bias):
    s = SHAPES[case["shape"]]
    T, E, K = case["T"], s["E"], s["K"]
    lg = logits.double()
    if not s["grouped"]:
        w, ids = torch.softmax(lg, 1).topk(K, 1)
        return ids, w / w.sum(1, keepdim=True)
    p = torch.sigmoid(lg)
    sel = p + bias.double()
    best = sel.view(T, 8, E // 8).topk(2, 2).values.sum(2).topk(4, 1).indices
    keep = torch.zeros((T, 8), dtype=torch.bool, device=lg.device).scatter_(1, best, True)
    ids = sel.masked_fill(~keep.repeat_interleave(E // 8, 1), -1e9).topk(K, 1).indices
    w = p.gather(1, ids)
    return ids, w / w.sum(1, keepdim=True) * 2.5


def exact(case, seed):
    s = SHAPES[case["shape"]]
    I, E = s["I"], s["E"]
    res = []
    for l in range(case["layers"]):
        gen = _generator(seed, l)
        x, logits, bias = _tokens(case, gen)
        ids, wts = _route(case, logits, bias)
        x = x.double()
        out = torch.zeros_like(x)
        e = 0
        for c13, s13, g13, c2, s2, g2 in _planes(case, gen):
            for j in range(c13.shape[0]):
                at = slice(j, j + 1)
                if e < E:
                    tok, k = (ids == e).nonzero(as_tuple=True)
                    w = wts[tok, k]
                else:
                    tok = torch.arange(case["T"], device=DEV)
                    w = torch.ones(case["T"], dtype=torch.float64, device=DEV)
                e += 1
                if tok.numel() == 0:
                    continue
                sub = lambda t: None if t is None else t[at]
                rows = x[tok]
                if case["int8"]:
                    rows = _int8_rows(rows)
                gu = rows @ _dequantize(case["fmt"], c13[at], sub(s13), sub(g13))[0].t()
                g, u = gu[:, :I], gu[:, I:]
                if s["limit"]:
                    g, u = g.clamp(max=s["limit"]), u.clamp(-s["limit"], s["limit"])
                act = g * torch.sigmoid(g) * u
                if case["int8"]:   # the int8 steps are of the bf16 rows
                    act = _int8_rows(act.to(torch.bfloat16).double())
                y = act @ _dequantize(case["fmt"], c2[at], sub(s2), sub(g2))[0].t()
                out.index_add_(0, tok, y * w[:, None])
        res.append({"out": out, "ids": ids.to(torch.int32), "weights": wts})
    return res
