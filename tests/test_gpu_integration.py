"""End-to-end GPU checks of the SGLang integration layer: EXL3LinearMethod and
EXL3MoEMethod built through create_weights -> checkpoint loaders ->
process_weights_after_loading -> apply, against the CPU oracle (bar:
max-abs-err <= 2e-2 * rms(ref), cosine >= 0.9999)."""

import numpy as np
import pytest
import torch
import torch.nn as nn

import oracle
from gpu_util import EXACT_WEIGHTS_REL, check_close, make_weight, make_x, product64, rel_error
from sglang_exl3 import ops
from sglang_exl3.exl3 import (
    MCG_MARKER_SIGNED_INT32,
    MUL1_MARKER_SIGNED_INT32,
    EXL3Config,
    EXL3MoEMethod,
    apply_exl3_experts,
)
from sglang_exl3.dense import EXL3DenseLinear, EXL3LinearMethod

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _registered():
    ops.register_custom_ops()


def _scaled(k, n, K, seed):
    tr, su, sv = make_weight(k, n, K, seed)
    return tr, su, (sv.astype(np.float32) * (4.0 / np.sqrt(k))).astype(np.float16)


@pytest.mark.parametrize("rows,shards,marker,cb,dtype", [
    (3, 2, "mcg", 1, torch.float16), (3, 3, "mul1", 2, torch.float16), (80, 2, "mcg", 1, torch.float16),
    (5, 1, None, 0, torch.float16), (1, 2, "mul1", 2, torch.float16), (80, 2, "mcg", 1, torch.bfloat16),
])
def test_linear_method_end_to_end(rows, shards, marker, cb, dtype):
    """fp16 layers are held to the bar; a bf16 layer's output is compared with
    the reference rounded to bf16 (its own rounding exceeds the bar at |y| ~ 20)."""
    print(f"case: linear rows={rows} shards={shards} cb={cb} {dtype}", flush=True)
    k, K = 256, 3
    outs = [256, 128, 128][:shards] if shards == 3 else [256] * shards
    method = EXL3LinearMethod(EXL3Config(bits=K, codebook="mul1" if marker == "mul1" else "mcg"), bits=K)
    layer = nn.Module()
    method.create_weights(layer, k, outs, k, sum(outs), dtype)
    weights = []
    for i, n in enumerate(outs):
        tr, su, sv = _scaled(k, n, K, seed=100 * rows + i)
        weights.append((tr, su, sv))
        p = lambda s: getattr(layer, f"exl3_{i}_{s}")
        method._load_linear(p("trellis"), torch.from_numpy(tr), i)
        method._load_linear(p("suh"), torch.from_numpy(su), i)
        method._load_linear(p("svh"), torch.from_numpy(sv), i)
        if marker:
            val = MCG_MARKER_SIGNED_INT32 if marker == "mcg" else MUL1_MARKER_SIGNED_INT32
            method._load_linear(p(marker), torch.tensor(val, dtype=torch.int32), i)
    method.process_weights_after_loading(layer)
    assert all(lin.codebook == cb for lin in layer._exl3_linears)
    x = make_x(rows, k, seed=rows)
    bias = np.random.default_rng(1).standard_normal(sum(outs)).astype(np.float32)
    y = method.apply(layer, torch.from_numpy(x).cuda().to(dtype).view(1, rows, k), torch.from_numpy(bias).cuda())
    torch.cuda.synchronize()
    assert y.shape == (1, rows, sum(outs)) and y.dtype == dtype
    x16 = torch.from_numpy(x).to(dtype).to(torch.float16).numpy()  # the input the layer saw, as fp16
    ref = np.concatenate([oracle.matmul(x16, oracle.dequant(tr, su, sv, K, cb, rtz=True)) for tr, su, sv in weights],
                         axis=1) + bias
    got = y.float().cpu().numpy().reshape(rows, -1)
    if dtype == torch.bfloat16:
        # bar + one bf16 ulp per element (output rounding of values near a boundary)
        ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref), 1e-30))) - 7)
        rms = float(np.sqrt(np.mean(ref.astype(np.float64) ** 2)))
        assert np.all(np.abs(got - ref) <= 2e-2 * rms + ulp)
        cos = float(np.dot(got.ravel(), ref.ravel()) / (np.linalg.norm(got) * np.linalg.norm(ref)))
        assert cos >= 0.9999
        return
    check_close(got, ref, f"linear method rows={rows}")


def _build_moe(E, hidden, inter, K, marker, seed):
    cfg = EXL3Config(bits=K, codebook=marker)
    method = EXL3MoEMethod(cfg, bits=K)
    layer = nn.Module()
    method.create_weights(layer, num_experts=E, hidden_size=hidden, intermediate_size_per_partition=inter,
                          params_dtype=torch.float16)
    layer.cuda()
    val = MCG_MARKER_SIGNED_INT32 if marker == "mcg" else MUL1_MARKER_SIGNED_INT32
    cb = 1 if marker == "mcg" else 2
    experts = []
    for e in range(E):
        spec = {}
        for j, (proj, shard, k, n) in enumerate((("gate", "w1", hidden, inter), ("up", "w3", hidden, inter),
                                                  ("down", "w2", inter, hidden))):
            tr, su, sv = _scaled(k, n, K, seed * 1000 + 3 * e + j)
            spec[proj] = (tr, su, sv, K, cb)
            pfx = "w13" if shard != "w2" else "w2"
            for suffix, arr in (("trellis", tr), ("suh", su), ("svh", sv)):
                method._load_exl3(getattr(layer, f"{pfx}_{suffix}"), torch.from_numpy(arr).cuda(),
                                  f"experts.{pfx}_{suffix}", shard_id=shard, expert_id=e)
            method._load_exl3(getattr(layer, f"{pfx}_{marker}"), torch.tensor(val, dtype=torch.int32),
                              f"experts.{pfx}_{marker}", shard_id=shard, expert_id=e)
        experts.append(spec)
    method.process_weights_after_loading(layer)
    return method, layer, experts


@pytest.mark.parametrize("T,topk,E,marker", [(1, 4, 8, "mcg"), (6, 2, 8, "mul1"), (20, 4, 16, "mcg")])
def test_moe_method_end_to_end(T, topk, E, marker):
    print(f"case: moe method T={T} topk={topk} E={E} {marker}", flush=True)
    hidden, inter, K = 256, 256, 3
    method, layer, experts = _build_moe(E, hidden, inter, K, marker, seed=T)
    rng = np.random.default_rng(T)
    ids = np.stack([rng.choice(E, topk, replace=False) for _ in range(T)]).astype(np.int64)
    w = rng.random((T, topk)).astype(np.float32)
    x = make_x(T, hidden, seed=T + 3)
    out = method.apply(layer, torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), torch.from_numpy(ids).cuda())
    torch.cuda.synchronize()
    assert layer._exl3_last_apply == "native"
    ref = oracle.moe_ref(x, ids, w, experts)
    check_close(out.float().cpu().numpy(), ref, "moe method native")
    # the eager per-expert loop over the same linears agrees too
    loop = apply_exl3_experts(torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda(),
                              layer, fused=False)
    torch.cuda.synchronize()
    assert layer._exl3_last_apply == "loop"
    check_close(loop.float().cpu().numpy(), ref, "moe method loop")


def test_moe_method_expert_parallel_map():
    """Global ids mapped through expert_map; ids of other ranks are skipped."""
    E_local, hidden, inter, K = 4, 256, 128, 2
    method, layer, experts = _build_moe(E_local, hidden, inter, K, "mcg", seed=77)
    # 8 global experts, this rank owns globals 4..7 as locals 0..3
    layer.expert_map = torch.tensor([-1, -1, -1, -1, 0, 1, 2, 3], dtype=torch.long)
    ids = np.array([[4, 1], [7, 5], [0, 2]], dtype=np.int64)
    w = np.array([[0.5, 0.5], [0.25, 0.75], [1.0, 1.0]], dtype=np.float32)
    x = make_x(3, hidden, seed=9)
    out = method.apply(layer, torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), torch.from_numpy(ids).cuda())
    torch.cuda.synchronize()
    local = np.where(ids >= 4, ids - 4, -1)
    ref = oracle.moe_ref(x, local, w, experts)
    o = out.float().cpu().numpy()
    assert np.all(o[2] == 0.0)
    check_close(o, ref, "moe expert map")


def test_dense_linear_forward_3inst():
    tr, su, sv = _scaled(256, 256, 4, seed=5)
    lin = EXL3DenseLinear(torch.from_numpy(tr).cuda(), torch.from_numpy(su).cuda(), torch.from_numpy(sv).cuda())
    x = make_x(2, 256, seed=2)
    y = lin.forward(torch.from_numpy(x).cuda(), {}, out_dtype=torch.float32)
    torch.cuda.synchronize()
    check_close(y.cpu().numpy(), oracle.matmul(x, oracle.dequant(tr, su, sv, 4, 0, rtz=True)), "3inst linear")


def test_moe_method_prefill_batch_stays_native():
    """A 2048-token top-8 batch (16384 routed rows) runs the device-side prefill
    pipeline through EXL3MoEMethod.apply, never the host-synced loop."""
    T, topk, E, hidden, inter, K = 2048, 8, 16, 256, 128, 3
    method, layer, experts = _build_moe(E, hidden, inter, K, "mul1", seed=99)
    rng = np.random.default_rng(98)
    ids = np.stack([rng.choice(E, topk, replace=False) for _ in range(T)]).astype(np.int64)
    w = rng.random((T, topk)).astype(np.float32)
    x = make_x(T, hidden, seed=97)
    out = method.apply(layer, torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), torch.from_numpy(ids).cuda())
    torch.cuda.synchronize()
    assert layer._exl3_last_apply == "native"
    sel = np.sort(rng.choice(T, 48, replace=False))
    check_close(out.float().cpu().numpy()[sel], oracle.moe_ref(x[sel], ids[sel], w[sel], experts), "moe prefill method")


@pytest.mark.parametrize("rows", [1, 5, 80])
def test_checkpoint_to_forward(tmp_path, rows):
    """A two-shard safetensors checkpoint streamed (iter_safetensors_pread) and routed
    (route_exl3_sidecar: fused qkv group cut into q/k/v shards, gate/up merged) into
    EXL3LinearMethod layers on the device; each layer's apply() against the oracle on the
    checkpoint's own groups."""
    from test_loader_sidecar import build_checkpoint, load_layers

    files, groups, dims = build_checkpoint(tmp_path)
    layers, leftovers = load_layers(files, dims)
    assert leftovers == ["model.norm.weight"]
    cfg = EXL3Config.from_config({"bits": 3, "codebook": "mcg"})

    def ref(x, mods):
        outs = []
        for mod in mods:
            t, su, sv = (a.numpy() for a in groups[mod])
            outs.append(oracle.matmul(x, oracle.dequant(t.view(np.int16), su, sv, 3, 1, rtz=True)))
        return np.concatenate(outs, axis=1)

    cases = {
        "model.layers.0.self_attn.qkv_proj": ["model.layers.0.self_attn.qkv_proj"],
        "model.layers.0.self_attn.o_proj": ["model.layers.0.self_attn.o_proj"],
        "model.layers.0.mlp.gate_up_proj": ["model.layers.0.mlp.gate_proj", "model.layers.0.mlp.up_proj"],
    }
    for prefix, mods in cases.items():
        layer = layers[prefix]
        method = EXL3LinearMethod(cfg, bits=3)
        method.process_weights_after_loading(layer)
        assert all(lin.trellis.is_cuda for lin in layer._exl3_linears)
        k = layer._exl3_lin_input_size_per_partition
        x = make_x(rows, k, seed=rows + len(prefix))
        y = method.apply(layer, torch.from_numpy(x).cuda().to(torch.bfloat16))
        torch.cuda.synchronize()
        assert y.dtype == torch.float16  # the layer's params dtype
        xr = torch.from_numpy(x).to(torch.bfloat16).to(torch.float16).numpy()
        check_close(y.float().cpu().numpy(), ref(xr, mods), f"checkpoint {prefix} rows={rows}")


@pytest.mark.parametrize("rows,n0,n1,K0,K1,cb0,cb1,second", [
    (1, 256, 256, 3, 3, 1, 1, False),     # (q, g): one batched launch on a shared input
    (4, 384, 384, 4, 4, 2, 2, True),      # (k, v) with a value residual: per-linear inputs, one launch
    (8, 256, 128, 3, 3, 1, 1, True),      # unequal widths: two launches
    (2, 256, 256, 3, 2, 1, 1, False),     # different K: two launches
    (3, 256, 256, 3, 3, 1, 2, True),      # different codebooks: two launches
    (80, 256, 256, 3, 3, 2, 2, True),     # above the batched row limit: two launches
])
def test_mgemm_two(rows, n0, n1, K0, K1, cb0, cb1, second):
    """_mgemm_two (reference dense.py:89-117): (x @ W0, x_b @ W1) against the oracle."""
    from sglang_exl3.dense import _mgemm_pair_compatible, _mgemm_two

    k = 256
    w0, w1 = _scaled(k, n0, K0, seed=40 + rows), _scaled(k, n1, K1, seed=41 + rows)
    mk = {1: torch.tensor([1], dtype=torch.int32), 2: None}
    mu = {1: None, 2: torch.tensor([1], dtype=torch.int32)}
    lins = [EXL3DenseLinear(*(torch.from_numpy(a).cuda() for a in w), mcg=mk[cb], mul1=mu[cb])
            for w, cb in ((w0, cb0), (w1, cb1))]
    assert _mgemm_pair_compatible(*lins) == (n0 == n1 and K0 == K1 and cb0 == cb1)
    x = make_x(rows, k, seed=50 + rows)
    xb = make_x(rows, k, seed=60 + rows) if second else None
    layer = nn.Module()
    y0, y1 = _mgemm_two(layer, torch.from_numpy(x).cuda(), *lins,
                        x2_b=None if xb is None else torch.from_numpy(xb).cuda())
    torch.cuda.synchronize()
    assert y0.shape == (rows, n0) and y1.shape == (rows, n1) and y0.dtype == y1.dtype == torch.float16
    ref0 = oracle.matmul(x, oracle.dequant(*w0, K0, cb0, rtz=True))
    ref1 = oracle.matmul(x if xb is None else xb, oracle.dequant(*w1, K1, cb1, rtz=True))
    check_close(y0.float().cpu().numpy(), ref0, f"mgemm first rows={rows}")
    check_close(y1.float().cpu().numpy(), ref1, f"mgemm second rows={rows}")
    # fresh outputs on every call
    z0, _ = _mgemm_two(layer, torch.from_numpy(x).cuda(), *lins,
                       x2_b=None if xb is None else torch.from_numpy(xb).cuda())
    assert z0.data_ptr() != y0.data_ptr() and torch.equal(z0, y0)


@pytest.mark.parametrize("m,widths,K,cb,x_dtype,y_dtype,env", [
    (1, (256, 128, 128), 4, 1, torch.bfloat16, torch.bfloat16, {}),   # balanced GEMV
    (3, (128, 384), 3, 2, torch.bfloat16, torch.float16, {}),         # ... two rows of blocks, mul1
    (5, (256, 128), 4, 0, torch.float16, torch.bfloat16, {}),         # k-split GEMV, fixed-point hand-off
    (11, (128, 256, 128, 128), 2, 1, torch.bfloat16, torch.bfloat16, {}),  # k-split GEMV, partial tiles
    # 16-row tiles, raw entries: finish launch, hand-off in the kernel, unsplit
    (14, (384, 128), 3, 2, torch.bfloat16, torch.bfloat16, {"EXL3_FAT_TALL": "0"}),
    (14, (384, 128), 3, 2, torch.bfloat16, torch.bfloat16, {"EXL3_FAT_TALL": "0", "EXL3_FAT_SPLIT_OUT": "0"}),
    (16, (256, 128), 5, 2, torch.float16, torch.bfloat16, {"EXL3_FAT_TALL": "0", "EXL3_FAT_HANDOFF": "0"}),
    (16, (256,), 3, 1, torch.float16, torch.bfloat16, {"EXL3_FAT_TALL": "0", "EXL3_FAT_HANDOFF": "0"}),  # fp32 sums, then bf16
    (13, (4096, 128, 256), 4, 0, torch.bfloat16, torch.bfloat16, {}),  # ... by default above 4096 columns, decoded values
    (14, (384, 128), 3, 2, torch.bfloat16, torch.bfloat16, {}),       # tall tiles from 13 rows, raw entries
    (40, (128, 256), 4, 1, torch.bfloat16, torch.float16, {}),        # tall tiles, finish launch
    (300, (256, 128), 3, 2, torch.bfloat16, torch.bfloat16, {"EXL3_FAT_TALL": "256", "EXL3_FAT_SPLITS": "1"}),  # no splits
    (70, (128, 256), 5, 2, torch.float16, torch.bfloat16, {"EXL3_FAT_HANDOFF": "0"}),  # the switches of other kernels
    (300, (256, 512), 3, 1, torch.bfloat16, torch.bfloat16, {"EXL3_FAT_WIDE": "2"}),   # name one weight's (tall tiles here)
])
def test_linear_cat(m, widths, K, cb, x_dtype, y_dtype, env, monkeypatch):
    """Several weights in one call, each kernel path, against one exl3_linear per weight with the casts
    around it.  The two only differ in the order of fp32 sums over k (other splits), so an element is at most
    a few roundings of the output type apart; twice for the clean-workspace contract."""
    for key, v in env.items():
        monkeypatch.setenv(key, v)
    k = 2048
    packs = [[torch.from_numpy(a).cuda() for a in _scaled(k, n, K, seed=7 * i + m)] for i, n in enumerate(widths)]
    x = torch.from_numpy(make_x(m, k, seed=m)).cuda().to(x_dtype)
    ref = torch.cat([torch.ops.sglang_exl3.exl3_linear(x.to(torch.float16), *p, K, cb) for p in packs], dim=1)
    ref = ref.to(y_dtype).float()
    for _ in range(2):
        y = torch.ops.sglang_exl3.exl3_linear_cat(x, *map(list, zip(*packs)), K, cb, y_dtype == torch.bfloat16)
        assert y.shape == ref.shape and y.dtype == y_dtype
        # one ulp of the output type, plus the fp32 sums' own error near zero
        ulp = 2.0 ** (-7 if y_dtype == torch.bfloat16 else -10)
        rms = float(ref.square().mean().sqrt())
        assert torch.all((y.float() - ref).abs() <= ulp * ref.abs() + 1e-3 * rms)


def _linear_layer(outs, k, K, cb, dtype, seed):
    """An EXL3LinearMethod layer of seeded shards, and the shards on the device."""
    method = EXL3LinearMethod(EXL3Config(bits=K, codebook="mul1" if cb == 2 else "mcg"), bits=K)
    layer = nn.Module()
    method.create_weights(layer, k, outs, k, sum(outs), dtype)
    packs = []
    for i, n in enumerate(outs):
        pack = [torch.from_numpy(a).cuda() for a in _scaled(k, n, K, seed=seed + i)]
        packs.append(pack)
        for suffix, t in zip(("trellis", "suh", "svh"), pack):
            method._load_linear(getattr(layer, f"exl3_{i}_{suffix}"), t, i)
        if cb:
            marker = "mcg" if cb == 1 else "mul1"
            val = MCG_MARKER_SIGNED_INT32 if cb == 1 else MUL1_MARKER_SIGNED_INT32
            method._load_linear(getattr(layer, f"exl3_{i}_{marker}"), torch.tensor(val, dtype=torch.int32), i)
    method.process_weights_after_loading(layer)
    return method, layer, packs


@pytest.mark.parametrize("rows,outs,cb,exact", [
    (8, [256, 256], 1, (0, 1)),
    (13, [256, 256], 1, (0, 1)),              # a pair keeps the pair form to 64 rows
    (64, [384, 384], 1, (0, 1)),
    (13, [512, 128, 128], 1, (1, 2)), (40, [512, 128, 128], 1, (1, 2)),
    (12, [8192, 4096], 1, (0, 1)),            # a sum of widths from 12288 on, each shard below it
    (9, [4096, 4096, 4096, 128], 0, (0, 1, 2, 3)),
    (12, [12288, 256], 1, (1,)),
    (8, [24576, 128], 1, (1,)),
    (16, [256, 256], 2, (0, 1)), (40, [512, 128, 128], 2, (0, 1, 2)), (12, [8192, 4096], 2, (0, 1)),
])
def test_linear_layer_weights_are_not_rounded(rows, outs, cb, exact):
    """Shards that separate calls and the batched launch multiply by exact codebook values (the pair-form GEMV, mul1's
    raw entries) have them in the one call too, for fp16 outputs where it shows."""
    print(f"case: exact weights rows={rows} outs={outs} cb={cb}", flush=True)
    k, K = 1024, 3
    method, layer, packs = _linear_layer(outs, k, K, cb, torch.float16, seed=rows)
    x = torch.from_numpy(make_x(rows, k, seed=rows)).cuda()
    got = method.apply(layer, x).split(outs, dim=1)
    for i in exact:
        err = rel_error(got[i], product64(x, *packs[i], K, cb))
        print(f"shard {i}: {err:.2e}", flush=True)
        assert err < EXACT_WEIGHTS_REL


@pytest.mark.parametrize("outs,cb,dtype", [
    ([512, 128, 128], 1, torch.bfloat16), ([512, 128, 128], 2, torch.float16), ([384, 256, 128], 0, torch.bfloat16),
    ([4096, 128, 256], 2, torch.bfloat16),
])
def test_kv_only_has_the_bits_of_apply(outs, cb, dtype):
    """apply_kv_only returns apply's K and V, packed, at every row count: GEMV plans, 16-row and tall tiles with and
    without k-splits, the batched pair (MCG, 13 to 64 rows)."""
    k, K = 2048, 3
    method, layer, packs = _linear_layer(outs, k, K, cb, dtype, seed=11)
    for rows in (1, 2, 4, 7, 11, 12, 13, 16, 17, 40, 64, 65, 200, 600):
        print(f"case: kv only outs={outs} cb={cb} rows={rows}", flush=True)
        x = torch.from_numpy(make_x(rows, k, seed=rows)).cuda().to(dtype).view(1, rows, k)
        want = method.apply(layer, x).split(outs, dim=-1)[1:]
        got = method.apply_kv_only(layer, x)
        for g, w in zip(got, want):
            assert g.is_contiguous() and g.dtype == dtype and torch.equal(g, w)
        # the operators themselves, from every weight on
        args = (x.view(rows, k), *map(list, zip(*packs)), K, cb, dtype == torch.bfloat16)
        cat = torch.ops.sglang_exl3.exl3_linear_cat(*args).split(outs, dim=1)
        for first in range(len(outs)):
            part = torch.ops.sglang_exl3.exl3_linear_part(*args, first).split([rows * n for n in outs[first:]])
            for p, c in zip(part, cat[first:]):
                assert torch.equal(p.view(rows, -1), c), (rows, first)
    assert method.apply_kv_only(layer, x[:, :0])[0].shape == (1, 0, outs[1])


@pytest.mark.parametrize("T,invalid", [(1, 0), (1, 1), (6, 2), (60, 0), (200, 3)])
def test_moe_bf16_matches_casts(T, invalid):
    """bf16 rows in and out of the one-call layer: the bits of the fp16 layer with casts around it (one token
    without routing, routed with the fused combine, with the combine launch, prefill), ids outside the
    experts included."""
    method, layer, _ = _build_moe(8, 256, 256, 3, "mcg", seed=T)
    g = torch.Generator().manual_seed(T)
    x = torch.randn((T, 256), generator=g).cuda().to(torch.bfloat16)
    ids = torch.stack([torch.randperm(8, generator=g)[:2] for _ in range(T)]).to(torch.int32).cuda()
    for j in range(invalid):
        ids[j % T, j % 2] = (-1, 8, 1 << 30)[j]
    w = torch.rand((T, 2), generator=g).cuda()
    got = method.apply(layer, x, w, ids)
    want = method.apply(layer, x.to(torch.float16), w, ids.to(torch.long)).to(torch.bfloat16)
    assert got.dtype == torch.bfloat16 and torch.equal(got, want)
