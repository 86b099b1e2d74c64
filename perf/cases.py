"""The work that users of this framework have it do, as timed cases.

Four kinds of case, each through the entry points a program calls:

* ``linear``: one quantized linear layer, ``EXL3LinearMethod.apply`` on a layer
  loaded through its own weight loaders (1 to 3 output shards, the model's
  dtype in and out), called eagerly as a prefill step calls it.
* ``op``: one registered operator (``torch.ops.sglang_exl3.*``) called eagerly:
  the bs=1 GEMV, the fused gate/up + SwiGLU, the whole-weight dequant.
* ``block``: the linears of dense decoder layers (qkv, o, gate/up + SwiGLU,
  down) for a decode batch, captured once in a HIP graph and replayed, which is
  how a server runs decode.
* ``moe``: routed-expert layers (``EXL3MoEMethod.apply``), replayed from a HIP
  graph for decode batches and called eagerly for prefill.

Weights are seeded random trellis words with +-1 input signs and output scales
that keep activations O(1); activations are N(0, 1).
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang-exl3_amd"))

from sglang_exl3 import exl3 as _exl3  # noqa: E402
from sglang_exl3.dense import EXL3LinearMethod  # noqa: E402
from sglang_exl3.ops import register_custom_ops  # noqa: E402

CODEBOOKS = ("3inst", "mcg", "mul1")
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}


# ------------------------------------------------------------------- the cases

def listed():
    return [
        # the headline call: one token through an 8B-class MLP projection
        {"name": "gemv-1", "kind": "op", "op": "exl3_gemv", "m": 1, "k": 4096, "n": 14336, "K": 4, "cb": "mcg"},
        # the smallest calls: qkv of a 1-2B model for one token, eager
        {"name": "qkv-small-1", "kind": "linear", "m": 1, "k": 2048, "shards": "2048,512,512", "K": 4, "cb": "mcg",
         "dtype": "bfloat16"},
        # qkv for a short ragged prompt or a speculative verification batch
        {"name": "qkv-77", "kind": "linear", "m": 77, "k": 4096, "shards": "4096,1024,1024", "K": 4, "cb": "mcg",
         "dtype": "bfloat16"},
        # down projection in a prefill chunk
        {"name": "down-1000", "kind": "linear", "m": 1000, "k": 14336, "shards": "4096", "K": 4, "cb": "mcg",
         "dtype": "bfloat16"},
        # fused gate/up of a prefill chunk, compute bound
        {"name": "gate-up-2048", "kind": "op", "op": "exl3_gate_up_swiglu", "m": 2048, "k": 4096, "n": 14336, "K": 3,
         "cb": "mul1"},
        # whole-weight decode (absorbing a weight, exporting it)
        {"name": "dequant", "kind": "op", "op": "dequant_trellis", "m": 1, "k": 4096, "n": 14336, "K": 4, "cb": "mcg"},
        # dense decode, a small batch
        {"name": "block-3", "kind": "block", "m": 3, "k": 4096, "kv": 1024, "n": 14336, "K": 4, "cb": "mcg",
         "layers": 2, "dtype": "float16"},
        # dense decode, a busy server
        {"name": "block-24", "kind": "block", "m": 24, "k": 4096, "kv": 1024, "n": 14336, "K": 3, "cb": "mul1",
         "layers": 2, "dtype": "bfloat16"},
        # sparse decode, one user
        {"name": "moe-1", "kind": "moe", "m": 1, "experts": 128, "topk": 8, "hidden": 2048, "inter": 768, "K": 3,
         "cb": "mcg", "skew": 1.1, "layers": 8, "graph": True, "dtype": "bfloat16"},
        # sparse decode, a busy server (skewed router)
        {"name": "moe-40", "kind": "moe", "m": 40, "experts": 128, "topk": 8, "hidden": 2048, "inter": 768, "K": 3,
         "cb": "mcg", "skew": 1.1, "layers": 4, "graph": True, "dtype": "bfloat16"},
        # a very wide expert layer: 288 routed experts, decode of four tokens
        {"name": "moe-wide-4", "kind": "moe", "m": 4, "experts": 288, "topk": 8, "hidden": 4096, "inter": 1536, "K": 3,
         "cb": "mul1", "skew": 0.0, "layers": 1, "graph": True, "dtype": "bfloat16"},
        # sparse prefill chunk
        {"name": "moe-2048", "kind": "moe", "m": 2048, "experts": 128, "topk": 8, "hidden": 2048, "inter": 768, "K": 3,
         "cb": "mcg", "skew": 1.1, "layers": 1, "graph": False, "dtype": "bfloat16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    return max(1, int(round(_log(rng, lo, hi) / 128))) * 128


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / 1e15)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("linear", "linear", "op", "block", "moe", "moe"))
        K, cb = rng.choice((2, 3, 3, 4, 4, 5, 6)), rng.choice(("mcg", "mul1"))
        dtype = rng.choice(("float16", "bfloat16", "bfloat16"))
        if kind == "linear":
            shards = [_width(rng, 256, 16384)]
            if rng.random() < 0.5:
                shards += [max(128, shards[0] // 4 // 128 * 128)] * 2
            case = {"kind": kind, "m": _log(rng, 1, 4096), "k": _width(rng, 512, 16384),
                    "shards": ",".join(map(str, shards)), "K": K, "cb": rng.choice((cb, cb, cb, "3inst")),
                    "dtype": dtype}
        elif kind == "op":
            op = rng.choice(("exl3_gemv", "exl3_gate_up_swiglu", "exl3_gate_up_swiglu", "dequant_trellis"))
            m = {"exl3_gemv": _log(rng, 1, 8), "exl3_gate_up_swiglu": _log(rng, 1, 2048), "dequant_trellis": 1}[op]
            case = {"kind": kind, "op": op, "m": m, "k": _width(rng, 1024, 8192), "n": _width(rng, 1024, 16384),
                    "K": K, "cb": cb}
        elif kind == "block":
            k = _width(rng, 2048, 6144)
            case = {"kind": kind, "m": _log(rng, 1, 48), "k": k, "kv": max(128, k // 4 // 128 * 128),
                    "n": _width(rng, 2 * k, 4 * k), "K": K, "cb": cb, "layers": 2, "dtype": dtype}
        else:
            m = _log(rng, 1, 2048)
            graph = m <= 64
            case = {"kind": kind, "m": m, "experts": rng.choice((16, 32, 60, 64, 128, 160)),
                    "topk": rng.choice((2, 4, 6, 8)), "hidden": _width(rng, 1024, 4096), "inter": _width(rng, 512, 1536),
                    "K": K, "cb": cb, "skew": rng.choice((0.0, 0.8, 1.1)), "layers": 2 if graph else 1,
                    "graph": graph, "dtype": dtype}
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ inputs

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + salt)
    return g


def _signs(g, *shape, scale=1.0):
    return ((torch.randint(0, 2, shape, device="cuda", generator=g) * 2 - 1) * scale).half()


def _words(g, *shape):
    return torch.randint(-32768, 32768, shape, dtype=torch.int16, device="cuda", generator=g)


def _pack(g, k, n, K):
    """(trellis, suh, svh) of one weight; svh carries 1/sqrt(k) so that outputs are O(1)."""
    return _words(g, k // 16, n // 16, 16 * K), _signs(g, k), _signs(g, n, scale=1.0 / math.sqrt(k))


def _rows(g, m, k, dtype):
    return torch.randn((m, k), dtype=torch.float32, device="cuda", generator=g).to(dtype)


def _shards(case):
    return [int(v) for v in case["shards"].split(",")]


def _linear_inputs(case, seed):
    g = _gen(seed)
    x = _rows(g, case["m"], case["k"], DTYPES[case["dtype"]])
    return x, [_pack(g, case["k"], n, case["K"]) for n in _shards(case)]


def _op_inputs(case, seed):
    g = _gen(seed)
    x = _rows(g, case["m"], case["k"], torch.float16)
    a = _pack(g, case["k"], case["n"], case["K"])
    return x, a, _pack(g, case["k"], case["n"], case["K"]) if case["op"] == "exl3_gate_up_swiglu" else None


def _block_inputs(case, seed):
    k, kv, n, K, dt = case["k"], case["kv"], case["n"], case["K"], DTYPES[case["dtype"]]
    out = []
    for i in range(case["layers"]):
        g = _gen(seed, i)
        out.append(SimpleNamespace(
            x=_rows(g, case["m"], k, dt), attn=_rows(g, case["m"], k, dt), x2=_rows(g, case["m"], k, dt),
            qkv=[_pack(g, k, w, K) for w in (k, kv, kv)], o=[_pack(g, k, k, K)], gate=_pack(g, k, n, K),
            up=_pack(g, k, n, K), down=[_pack(g, n, k, K)]))
    return out


def _routing(case, seed):
    """Top-k of softmax(N(0,1) + log p), p ~ rank^-skew over a seeded permutation, weights renormalised."""
    rng = np.random.default_rng(seed)
    e = case["experts"]
    p = (np.arange(1, e + 1, dtype=np.float64) ** -case["skew"])[rng.permutation(e)]
    z = rng.standard_normal((case["m"], e)) + np.log(p / p.sum())
    ids = np.argsort(-z, axis=1)[:, :case["topk"]]
    w = np.exp(np.take_along_axis(z, ids, axis=1))
    return ids.astype(np.int32), (w / w.sum(axis=1, keepdims=True)).astype(np.float32)


def _moe_inputs(case, seed):
    e, h, i, kw = case["experts"], case["hidden"], case["inter"], 16 * case["K"]
    out = []
    for layer in range(case["layers"]):
        g = _gen(seed, layer)
        ids, w = _routing(case, int(seed) * 64 + layer)
        out.append(SimpleNamespace(
            x=_rows(g, case["m"], h, DTYPES[case["dtype"]]), ids=torch.from_numpy(ids).cuda(),
            w=torch.from_numpy(w).cuda(),
            w13_trellis=_words(g, e, 2, h // 16, i // 16, kw), w13_suh=_signs(g, e, 2, h),
            w13_svh=_signs(g, e, 2, i, scale=1.0 / math.sqrt(h)),
            w2_trellis=_words(g, e, i // 16, h // 16, kw), w2_suh=_signs(g, e, i),
            w2_svh=_signs(g, e, h, scale=1.0 / math.sqrt(i))))
    return out


# ------------------------------------------------------- layers as a server loads them

def _linear_layer(packs, k, K, cb, dtype):
    method = EXL3LinearMethod(SimpleNamespace(bits=K), bits=K)
    layer = torch.nn.Module()
    sizes = [int(p[2].numel()) for p in packs]
    method.create_weights(layer, k, sizes, k, sum(sizes), dtype)
    for i, pack in enumerate(packs):
        for suffix, t in zip(("trellis", "suh", "svh"), pack):
            p = getattr(layer, f"exl3_{i}_{suffix}")
            p.weight_loader(p, t, i)
        if cb != "3inst":
            p = getattr(layer, f"exl3_{i}_{cb}")
            p.weight_loader(p, torch.ones(1, dtype=torch.int32), i)
    method.process_weights_after_loading(layer)
    return lambda x: method.apply(layer, x)


def _moe_layer(case, inp):
    method = _exl3.EXL3MoEMethod(SimpleNamespace(bits=case["K"], codebook=case["cb"]), bits=case["K"])
    layer = torch.nn.Module()
    with torch.device("cuda"):
        method.create_weights(layer, case["experts"], case["hidden"], case["inter"], inp.x.dtype)
    for name in ("w13_trellis", "w13_suh", "w13_svh", "w2_trellis", "w2_suh", "w2_svh"):
        getattr(layer, name).data.copy_(getattr(inp, name))
        delattr(inp, name)
    for name in ("w13_", "w2_"):
        getattr(layer, name + case["cb"]).data.fill_(1)
    method.process_weights_after_loading(layer)
    return lambda: method.apply(layer, inp.x, inp.w, inp.ids)


_STREAM = None


def _captured(step):
    """`step` as a HIP graph: one warm-up on the capture stream, then the capture.  The replay holds
    `step`, and with it the weights and inputs whose addresses the graph recorded."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    _STREAM.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_STREAM):
        step()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=_STREAM):
            out = step()
    torch.cuda.current_stream().wait_stream(_STREAM)

    def replay(held=step):
        graph.replay()
        return out

    return replay


def prepare(case, seed):
    register_custom_ops()
    ops = torch.ops.sglang_exl3
    K, cb = case["K"], CODEBOOKS.index(case["cb"])
    if case["kind"] == "linear":
        x, packs = _linear_inputs(case, seed)
        apply = _linear_layer(packs, case["k"], K, case["cb"], x.dtype)
        return lambda: apply(x)
    if case["kind"] == "op":
        x, a, b = _op_inputs(case, seed)
        if case["op"] == "exl3_gemv":
            return lambda: ops.exl3_gemv(x, *a, K, cb == 1)
        if case["op"] == "dequant_trellis":
            return lambda: ops.dequant_trellis(*a, K, cb == 1)
        return lambda: ops.exl3_gate_up_swiglu(x, a[1], a[0], a[2], b[0], b[2], K, cb)
    if case["kind"] == "block":
        steps = []
        for d in _block_inputs(case, seed):
            dt = d.x.dtype
            qkv = _linear_layer(d.qkv, case["k"], K, case["cb"], dt)
            o = _linear_layer(d.o, case["k"], K, case["cb"], dt)
            down = _linear_layer(d.down, case["n"], K, case["cb"], dt)
            steps.append((d, qkv, o, down))

        def block():
            out = []
            for d, qkv, o, down in steps:
                h = ops.exl3_gate_up_swiglu(d.x2.half(), d.gate[1], d.gate[0], d.gate[2], d.up[0], d.up[2], K, cb)
                out.append([qkv(d.x), o(d.attn), h, down(h)])
            return out

        return _captured(block)
    layers = [_moe_layer(case, inp) for inp in _moe_inputs(case, seed)]

    def moe():
        return [layer() for layer in layers]

    return _captured(moe) if case["graph"] else moe


def run(state):
    return state()


# ------------------------------------------------------------------- figures

def _mat(k, n, K):
    return k * n * K / 8 + 2 * (k + n)


def work(case):
    m, K = case["m"], case["K"]
    if case["kind"] == "linear":
        k, ns = case["k"], _shards(case)
        return {"bytes": sum(_mat(k, n, K) for n in ns) + 2 * m * (k + sum(ns)), "flops": 2.0 * m * k * sum(ns)}
    if case["kind"] == "op":
        k, n = case["k"], case["n"]
        if case["op"] == "dequant_trellis":
            return {"bytes": _mat(k, n, K) + 2.0 * k * n, "flops": 2.0 * 7 * 2 * k * n}
        p = 2 if case["op"] == "exl3_gate_up_swiglu" else 1
        return {"bytes": p * _mat(k, n, K) + 2 * m * (k + n), "flops": 2.0 * p * m * k * n}
    if case["kind"] == "block":
        k, kv, n = case["k"], case["kv"], case["n"]
        mats = [(k, k + 2 * kv), (k, k), (k, 2 * n), (n, k)]
        b = sum(_mat(a, c, K) for a, c in mats) + 2 * m * (3 * k + k + 2 * kv + k + n + k)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * sum(2.0 * m * a * c for a, c in mats)}
    h, i = case["hidden"], case["inter"]
    used = np.mean([len(np.unique(_routing(case, s)[0])) for s in range(3)])
    b = used * (2 * _mat(h, i, K) + _mat(i, h, K)) + 4 * m * h
    return {"bytes": case["layers"] * b, "flops": case["layers"] * 6.0 * m * case["topk"] * h * i}


def tolerance(case):
    if case["kind"] == "op" and case["op"] == "dequant_trellis":
        return "exact"
    # measured against exact(): 3e-4 to 6e-4 with fp16 outputs, 1.7e-3 to 1.8e-3 with bfloat16; four times that
    return {"rel": 7.2e-3 if case.get("dtype") == "bfloat16" else 2.4e-3}


# ------------------------------------------------------- the same in 64 bits, plain torch

def _codebook(cb):
    s = np.arange(65536, dtype=np.uint64)
    if cb == "mul1":
        x = (s * 0x83DCD12D) & 0xFFFFFFFF
        total = (x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + (x >> 24)
        half = np.array([0x1EEE, 0xC931], dtype=np.uint16).view(np.float16).astype(np.float64)
        return (1024.0 + total.astype(np.float64)) * half[0] + half[1]
    x = s * 89226354 + 64248484 if cb == "3inst" else s * 0xCBAC1FED
    x = ((x & 0x8FFF8FFF) ^ 0x3B603B60).astype(np.uint32)
    return x.view(np.float16).astype(np.float64).reshape(-1, 2).sum(axis=1)


def _hadamard():
    h = torch.ones((1, 1), dtype=torch.float64)
    while h.shape[0] < 128:
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return (h / math.sqrt(128.0)).cuda()


def _decoded(trellis, cb):
    """The rotated weight [k, n] in float64: 16-bit windows of each tile's MSB-first 32-bit words, through the codebook."""
    kt, nt, kw = trellis.shape
    K = kw // 16
    v = trellis.reshape(-1, kw // 2, 2).to(torch.int64) & 0xFFFF
    words = v[..., 0] | (v[..., 1] << 16)
    t = torch.arange(256, device="cuda")
    start = ((t + 257) * K - 16) % (256 * K)
    last = (start + 15) // 32
    pair = (words[:, start // 32] << 32) | words[:, last % (kw // 2)]
    state = (pair >> ((last + 1) * 32 - start - 16)) & 0xFFFF
    val = torch.from_numpy(_codebook(cb)).cuda()[state]
    lane, j = t >> 3, t & 7
    row = 2 * (lane & 3) + (j & 1) + 8 * ((j >> 1) & 1)
    col = (lane >> 2) + 8 * (j >> 2)
    tile = torch.empty_like(val)
    tile[:, row * 16 + col] = val
    return tile.view(kt, nt, 16, 16).permute(0, 2, 1, 3).reshape(kt * 16, nt * 16)


def _rotate(x, had):
    return (x.reshape(-1, 128) @ had).view(x.shape)


def _product(x, pack, cb, had):
    trellis, suh, svh = pack
    y = _rotate(x.double() * suh.double(), had) @ _decoded(trellis, cb)
    return _rotate(y, had) * svh.double()


def _swiglu(x, gate, up, cb, had):
    g, u = _product(x, gate, cb, had), _product(x, up, cb, had)
    return torch.nn.functional.silu(g) * u


def exact(case, seed):
    had, cb = _hadamard(), case["cb"]
    if case["kind"] == "linear":
        x, packs = _linear_inputs(case, seed)
        return torch.cat([_product(x, p, cb, had) for p in packs], dim=1)
    if case["kind"] == "op":
        x, a, b = _op_inputs(case, seed)
        if case["op"] == "exl3_gemv":
            return _product(x, a, cb, had)
        if case["op"] == "dequant_trellis":
            w = _rotate(_decoded(a[0], cb), had).t().contiguous()
            w = _rotate(w, had).t() * a[1].double()[:, None]
            return w * a[2].double()
        return _swiglu(x, a, (b[0], a[1], b[2]), cb, had)
    if case["kind"] == "block":
        out = []
        for d in _block_inputs(case, seed):
            h = _swiglu(d.x2, d.gate, (d.up[0], d.gate[1], d.up[2]), cb, had)
            out.append([torch.cat([_product(d.x, p, cb, had) for p in d.qkv], dim=1), _product(d.attn, d.o[0], cb, had),
                        h, _product(h, d.down[0], cb, had)])
        return out
    outs = []
    for d in _moe_inputs(case, seed):
        y = torch.zeros(d.x.shape, dtype=torch.float64, device="cuda")
        for e in torch.unique(d.ids).tolist():
            tok, slot = (d.ids == e).nonzero(as_tuple=True)
            gate, up = ((d.w13_trellis[e, p], d.w13_suh[e, p], d.w13_svh[e, p]) for p in (0, 1))
            h = _swiglu(d.x[tok], gate, up, cb, had)
            z = _product(h, (d.w2_trellis[e], d.w2_suh[e], d.w2_svh[e]), cb, had)
            y.index_add_(0, tok, z * d.w[tok, slot].double()[:, None])
        outs.append(y)
    return outs
