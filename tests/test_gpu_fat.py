"""GPU parity of the many-row MFMA GEMM: exl3_fat_gemm / exl3_fat_gemm_scatter
(rotated fp16 input, fp32 output) and exl3_gemm's prefill path (m ≥ 12),
against the oracle (bar: max-abs-err <= 2e-2 * rms(ref), cosine >= 0.9999)."""

import numpy as np
import pytest
import torch

import oracle
from gpu_util import check_close, make_weight, make_x
from sglang_exl3 import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _registered():
    ops.register_custom_ops()


def _rotate(x, suh):
    """fp16(H(x * suh) / sqrt(128)) per 128 block (the input the fat GEMM takes)."""
    return oracle.had_rows(x.astype(np.float32), suh, None, np.float32(0.08838834764831845)).astype(np.float16)


def _ref(a_rot, trellis, svh, K, cb):
    """svh * H(a_rot . T) / sqrt(128), with T the decoded tiles (no rotations)."""
    k, n = trellis.shape[0] * 16, trellis.shape[1] * 16
    ones_k = np.ones(k, dtype=np.float16)
    ones_n = np.ones(n, dtype=np.float16)
    # the oracle's dequant W = suh*svh*(H T H)/128; with unit scales, H W H = 128 T... use decode_tile directly
    T = np.zeros((k, n), dtype=np.float32)
    for kt in range(k // 16):
        for nt in range(n // 16):
            T[kt * 16:(kt + 1) * 16, nt * 16:(nt + 1) * 16] = oracle.f16_to_f32(
                oracle.decode_tile(trellis[kt, nt].view(np.uint16), K, cb, rtz=False))
    y = a_rot.astype(np.float64) @ T.astype(np.float64)
    del ones_k, ones_n
    return oracle.had_rows(y.astype(np.float32), None, svh, np.float32(0.08838834764831845))


@pytest.mark.parametrize("M,k,n,K,cb", [
    (16, 256, 256, 4, 1), (1, 256, 128, 3, 2), (40, 512, 384, 3, 1), (128, 256, 256, 4, 0),
    (200, 1024, 256, 2, 2), (300, 256, 512, 5, 1),
])
def test_fat_gemm_vs_oracle(M, k, n, K, cb):
    print(f"case: fat M={M} k={k} n={n} K={K} cb={cb}", flush=True)
    tr, su, sv = make_weight(k, n, K, seed=M * 13 + K)
    x = make_x(M, k, seed=M)
    a = _rotate(x, su)
    out = torch.full((M, n), 123.0, dtype=torch.float32, device="cuda")  # overwritten
    mcg, mul1 = cb == 1, cb == 2
    torch.ops.sglang_exl3.exl3_fat_gemm(torch.from_numpy(a).cuda(), torch.from_numpy(tr).cuda(), out,
                                        torch.from_numpy(sv).cuda(), K, mcg, mul1)
    torch.cuda.synchronize()
    check_close(out.cpu().numpy(), _ref(a, tr, sv, K, cb), f"fat M={M}")


def _with_env(name, value, fn):
    import os
    old = os.environ.get(name)
    os.environ[name] = value
    try:
        return fn()
    finally:
        if old is None:
            del os.environ[name]
        else:
            os.environ[name] = old


def _fat(a, tr, sv, K, cb, M, n):
    out = torch.full((M, n), 123.0, dtype=torch.float32, device="cuda")  # overwritten
    torch.ops.sglang_exl3.exl3_fat_gemm(torch.from_numpy(a).cuda(), torch.from_numpy(tr).cuda(), out,
                                        torch.from_numpy(sv).cuda(), K, cb == 1, cb == 2)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
def test_fat_wide_tiles_every_width(K, cb):
    """Wide-tile kernel (256 x 256 tiles, above 256 rows): every bit width and codebook,
    a partial second row tile (ending in the first row half), k-splits accumulating atomically."""
    M, k, n = 300, 256, 256
    print(f"case: fat wide M={M} k={k} n={n} K={K} cb={cb}", flush=True)
    tr, su, sv = make_weight(k, n, K, seed=100 + 3 * K + cb)
    a = _rotate(make_x(M, k, seed=K + 10 * cb), su)
    out = _with_env("EXL3_FAT_WIDE", "2", lambda: _fat(a, tr, sv, K, cb, M, n))
    check_close(out, _ref(a, tr, sv, K, cb), f"fat wide K={K} cb={cb}")


@pytest.mark.parametrize("M,k,n,K,cb", [(512, 1024, 512, 3, 2), (257, 512, 768, 4, 1), (65, 2048, 256, 2, 0),
                                        (1100, 128, 512, 5, 1)])
@pytest.mark.parametrize("wide", ["2", "1", "0"])
def test_fat_wide_and_narrow_kernels(M, k, n, K, cb, wide):
    """The same shapes through the wide-tile kernel (EXL3_FAT_WIDE=2), the
    default plan and the narrow kernel (EXL3_FAT_WIDE=0)."""
    print(f"case: fat M={M} k={k} n={n} K={K} cb={cb} wide={wide}", flush=True)
    tr, su, sv = make_weight(k, n, K, seed=M + n)
    a = _rotate(make_x(M, k, seed=M + 1), su)
    out = _with_env("EXL3_FAT_WIDE", wide, lambda: _fat(a, tr, sv, K, cb, M, n))
    check_close(out, _ref(a, tr, sv, K, cb), f"fat M={M} wide={wide}")


def test_fat_wide_scatter_accumulates(monkeypatch):
    monkeypatch.setenv("EXL3_FAT_WIDE", "2")  # the wide-tile kernel at this small grid
    M, k, n, K = 300, 512, 512, 3
    tr, su, sv = make_weight(k, n, K, seed=15)
    a = _rotate(make_x(M, k, seed=16), su)
    rng = np.random.default_rng(17)
    tok = rng.integers(0, 40, size=M).astype(np.int64)
    rw = (rng.random(M) + 0.5).astype(np.float16)
    base = rng.standard_normal((40, n)).astype(np.float32)
    out = torch.from_numpy(base.copy()).cuda()
    torch.ops.sglang_exl3.exl3_fat_gemm_scatter(torch.from_numpy(a).cuda(), torch.from_numpy(tr).cuda(), out,
                                                torch.from_numpy(sv).cuda(), torch.from_numpy(tok).cuda(),
                                                torch.from_numpy(rw).cuda(), K, False, True)
    torch.cuda.synchronize()
    rows = _ref(a, tr, sv, K, 2) * rw.astype(np.float32)[:, None]
    want = base.copy()
    np.add.at(want, tok, rows)
    check_close(out.cpu().numpy() - base, want - base, "fat wide scatter")


def test_fat_gemm_scatter_accumulates():
    M, k, n, K = 48, 256, 256, 4
    tr, su, sv = make_weight(k, n, K, seed=5)
    x = make_x(M, k, seed=6)
    a = _rotate(x, su)
    rng = np.random.default_rng(7)
    tok = rng.integers(0, 20, size=M).astype(np.int64)  # destinations repeat: atomics
    rw = (rng.random(M) + 0.5).astype(np.float16)
    base = rng.standard_normal((20, n)).astype(np.float32)
    out = torch.from_numpy(base.copy()).cuda()
    torch.ops.sglang_exl3.exl3_fat_gemm_scatter(torch.from_numpy(a).cuda(), torch.from_numpy(tr).cuda(), out,
                                                torch.from_numpy(sv).cuda(), torch.from_numpy(tok).cuda(),
                                                torch.from_numpy(rw).cuda(), K, True, False)
    torch.cuda.synchronize()
    rows = _ref(a, tr, sv, K, 1) * rw.astype(np.float32)[:, None]
    want = base.copy()
    np.add.at(want, tok, rows)
    check_close(out.cpu().numpy() - base, want - base, "fat scatter")


@pytest.mark.parametrize("m,k,n,K,cb", [(65, 256, 256, 4, 1), (200, 512, 384, 3, 2), (1000, 256, 128, 2, 1),
                                        (300, 128, 512, 3, 1), (700, 1024, 256, 4, 2)])
def test_gemm_prefill_path_vs_oracle(m, k, n, K, cb):
    print(f"case: gemm prefill m={m} k={k} n={n}", flush=True)
    tr, su, sv = make_weight(k, n, K, seed=m + k)
    x = make_x(m, k, seed=m)
    y = torch.ops.sglang_exl3.exl3_gemm(torch.from_numpy(x).cuda(), torch.from_numpy(tr).cuda(),
                                        torch.from_numpy(su).cuda(), torch.from_numpy(sv).cuda(), K, cb == 1)
    torch.cuda.synchronize()
    ref = oracle.matmul(x, oracle.dequant(tr, su, sv, K, cb, rtz=True))
    check_close(y.float().cpu().numpy(), ref, f"gemm prefill m={m}")


def test_fat_then_gemv_workspace_stays_clean():
    """The prefill scratch must not disturb the GEMV counters sharing the workspace."""
    k, n, K = 512, 1024, 4
    tr, su, sv = make_weight(k, n, K, seed=1)
    d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
    xb = make_x(300, k, seed=2)
    torch.ops.sglang_exl3.exl3_gemm(torch.from_numpy(xb).cuda(), *d, K, True)
    xs = make_x(2, k, seed=3)
    y = torch.ops.sglang_exl3.exl3_gemv(torch.from_numpy(xs).cuda(), *d, K, True, 1)
    torch.cuda.synchronize()
    check_close(y.float().cpu().numpy(), oracle.matmul(xs, oracle.dequant(tr, su, sv, K, 1, rtz=True)), "gemv after")


@pytest.mark.parametrize("cb", [1, 2])
@pytest.mark.parametrize("op", ["gemm", "gate_up"])
def test_tail_split_repeatable(op, cb, monkeypatch):
    """The last round's tiles in parts: of the wide-tile kernel (exl3_gemm, EXL3_FAT_WIDE=2) as two k-halves, the first
    half handing its sums to the second, of the fused gate/up kernel (EXL3_GU_TALL=1) as row parts.  Every tile of
    these one-round launches: against the oracle, bit-identical over repeated calls (the hand-off counts and flags
    reset themselves), and close to the launch of whole tiles (EXL3_FAT_TAIL=0)."""
    # gemm: 56 x 2 tiles, enough for one k-split (smaller grids split k with
    # fp32 atomics instead); gate/up: 2 x 2 tiles, always one split
    m, k, K = (512, 1024, 3) if op == "gemm" else (300, 1024, 3)
    n = 14336 if op == "gemm" else 256
    print(f"case: tail split {op} m={m} k={k} n={n} cb={cb}", flush=True)
    x = torch.from_numpy(make_x(m, k, seed=31)).cuda()
    if op == "gemm":
        monkeypatch.setenv("EXL3_FAT_WIDE", "2")
        tr, su, sv = make_weight(k, n, K, seed=32)
        d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
        run = lambda: torch.ops.sglang_exl3.exl3_gemm(x, *d, K, cb == 1)
        ref = oracle.matmul(x.cpu().numpy(), oracle.dequant(tr, su, sv, K, cb, rtz=True))
    else:
        monkeypatch.setenv("EXL3_GU_TALL", "1")
        tg, su, sg = make_weight(k, n, K, seed=33)
        tu, _, su2 = make_weight(k, n, K, seed=34)
        d = [torch.from_numpy(v).cuda() for v in (su, tg, sg, tu, su2)]
        run = lambda: torch.ops.sglang_exl3.exl3_gate_up_swiglu(x, *d, K, cb)
        g = oracle.matmul(x.cpu().numpy(), oracle.dequant(tg, su, sg, K, cb, rtz=True))
        u = oracle.matmul(x.cpu().numpy(), oracle.dequant(tu, su, su2, K, cb, rtz=True))
        ref = oracle.swiglu(g, u, float("inf"))
    outs = [run() for _ in range(3)]
    torch.cuda.synchronize()
    for o in outs[1:]:
        assert torch.equal(o, outs[0]), "tail split: repeated calls differ"
    check_close(outs[0].float().cpu().numpy(), ref, f"tail split {op}")
    monkeypatch.setenv("EXL3_FAT_TAIL", "0")
    whole = run()
    torch.cuda.synchronize()
    check_close(outs[0].float().cpu().numpy(), whole.float().cpu().numpy(), f"tail split vs whole {op}")
    if op == "gate_up":  # the same sums, other workgroups
        assert torch.equal(outs[0], whole)


@pytest.mark.parametrize("op,m", [("gemm", 16), ("gemm", 20), ("gemm", 48), ("gemm", 300), ("gate_up", 16), ("gate_up", 48),
                                  ("gate_up", 200)])
def test_mul1_raw_entries(op, m, monkeypatch):
    """Narrow 16-row MFMA tiles and tall tiles on mul1 weights read raw entries
    (1024 + byte sum, no affine step) and correct in the epilogue with kinv * acc
    + bias * (row sum of the rotated x over the split's k range).  k = 14336 (112
    chunk sums per row), 16-row tiles with k-splits (m = 16; EXL3_FAT_TALL=0 for
    gemm, which takes tall tiles there at this width), tall tiles (gemm m = 20,
    gate/up m = 48 and 200): against the oracle and close to the decoded path
    (EXL3_FAT_RAW=0).  The 64-row tiles (gemm m = 48, EXL3_FAT_TALL=0) and the
    plain wide tiles (gemm m = 300, EXL3_FAT_WIDE=2: 16 fp32-atomic k-splits)
    decode values and are checked at the same k."""
    k, n, K, cb = 14336, 256, 3, 2
    if op == "gemm" and m != 20:
        monkeypatch.setenv(*(("EXL3_FAT_WIDE", "2") if m > 256 else ("EXL3_FAT_TALL", "0")))
    print(f"case: raw mul1 {op} m={m} k={k} n={n}", flush=True)
    x = torch.from_numpy(make_x(m, k, seed=51 + m)).cuda()
    if op == "gemm":
        tr, su, sv = make_weight(k, n, K, seed=52)
        d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
        run = lambda: torch.ops.sglang_exl3.exl3_gemm(x, *d, K, False)
        ref = oracle.matmul(x.cpu().numpy(), oracle.dequant(tr, su, sv, K, cb, rtz=True))
    else:
        tg, su, sg = make_weight(k, n, K, seed=53)
        tu, _, su2 = make_weight(k, n, K, seed=54)
        # svh / 16 keeps silu(g) * u inside fp16 at this k
        sg, su2 = (sg / 16).astype(np.float16), (su2 / 16).astype(np.float16)
        d = [torch.from_numpy(v).cuda() for v in (su, tg, sg, tu, su2)]
        run = lambda: torch.ops.sglang_exl3.exl3_gate_up_swiglu(x, *d, K, cb)
        g = oracle.matmul(x.cpu().numpy(), oracle.dequant(tg, su, sg, K, cb, rtz=True))
        u = oracle.matmul(x.cpu().numpy(), oracle.dequant(tu, su, su2, K, cb, rtz=True))
        ref = oracle.swiglu(g, u, float("inf"))
    raw = run()
    torch.cuda.synchronize()
    check_close(raw.float().cpu().numpy(), ref, f"raw mul1 {op} m={m}")
    monkeypatch.setenv("EXL3_FAT_RAW", "0")
    dec = run()
    torch.cuda.synchronize()
    check_close(raw.float().cpu().numpy(), dec.float().cpu().numpy(), f"raw vs decoded {op} m={m}")


@pytest.mark.parametrize("mt", [128, 256])
@pytest.mark.parametrize("m,k,n,K,cb,splits", [
    (1, 128, 128, 4, 1, 1), (17, 256, 384, 1, 2, 2), (31, 512, 128, 2, 0, 4), (33, 1024, 256, 3, 2, 8),
    (64, 2048, 128, 4, 1, 16), (65, 256, 128, 5, 1, 1), (128, 512, 256, 6, 2, 2), (129, 384, 128, 7, 0, 1),
    (255, 1024, 128, 8, 1, 8), (256, 256, 384, 3, 1, 1), (257, 512, 128, 4, 2, 4), (700, 256, 128, 3, 0, 2)])
def test_tall_tiles(m, k, n, K, cb, splits, mt, monkeypatch):
    """Tall tiles of both heights at the edges of their 32-row groups and tiles, every K and codebook, with and
    without the finish launch: against the oracle, twice (nothing is left behind in the scratch), and an output
    that is only 4-byte aligned."""
    print(f"case: tall tiles mt={mt} m={m} k={k} n={n} K={K} cb={cb} splits={splits}", flush=True)
    monkeypatch.setenv("EXL3_FAT_TALL", str(mt))
    monkeypatch.setenv("EXL3_FAT_SPLITS", str(splits))
    monkeypatch.setenv("EXL3_GEMM_GEMV_ROWS", "0")
    tr, su, sv = make_weight(k, n, K, seed=m + K)
    x = make_x(m, k, seed=m)
    d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
    xd = torch.from_numpy(x).cuda()
    y = torch.ops.sglang_exl3.exl3_linear(xd, *d, K, cb)
    assert torch.equal(y, torch.ops.sglang_exl3.exl3_linear(xd, *d, K, cb))
    ref = oracle.matmul(x, oracle.dequant(tr, su, sv, K, cb, rtz=True))
    check_close(y.float().cpu().numpy(), ref, f"tall m={m}")
    lib = _lib.lib()
    need = lib.exl3_gemm_workspace_size(m, k, n, K)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    odd = torch.zeros(m * n + 2, dtype=torch.float16, device="cuda")
    rc = lib.exl3_gemm(xd.data_ptr(), *[t.data_ptr() for t in d], odd.data_ptr() + 4, m, k, n, K, cb, ws.data_ptr(),
                       need, int(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "exl3_gemm")
    assert torch.equal(odd[2:].view(m, n), y)


@pytest.mark.parametrize("few", ["0", "1000000"])
@pytest.mark.parametrize("m,k,cb", [(17, 384, 1), (33, 128, 2), (70, 1152, 2)])
def test_rotation_of_dword_aligned_rows(m, k, cb, few, monkeypatch):
    """Both input rotations (8 chunks a wave, one a wave) on x and suh that are only 4-byte aligned, with chunk counts
    that do not fill their waves or workgroups (51, 33, 630), and the chunk sums that mul1 tiles read: the aligned
    call's bits, fp16 and bf16."""
    n, K = 128, 4
    print(f"case: rotation alignment m={m} k={k} cb={cb} few={few}", flush=True)
    monkeypatch.setenv("EXL3_ROTATE_FEW", few)
    tr, su, sv = (torch.from_numpy(v).cuda() for v in make_weight(k, n, K, seed=m))
    xs = torch.from_numpy(make_x(m, k, seed=m)).cuda()
    su_odd = torch.zeros(k + 2, dtype=torch.float16, device="cuda")
    su_odd[2:] = su
    for dtype in (torch.float16, torch.bfloat16):
        x = xs.to(dtype)
        x_odd = torch.zeros(m * k + 2, dtype=dtype, device="cuda")
        x_odd[2:] = x.reshape(-1)
        cat = torch.ops.sglang_exl3.exl3_linear_cat
        want = cat(x, [tr], [su], [sv], K, cb, False)
        assert torch.equal(cat(x_odd[2:].view(m, k), [tr], [su_odd[2:]], [sv], K, cb, False), want)
    ref = oracle.matmul(xs.cpu().numpy(), oracle.dequant(*(t.cpu().numpy() for t in (tr, su, sv)), K, cb, rtz=True))
    check_close(cat(xs, [tr], [su], [sv], K, cb, False).float().cpu().numpy(), ref, f"rotation m={m} k={k}")


@pytest.mark.parametrize("m", [40, 200])
def test_tall_tiles_take_the_splits_that_fit(m):
    """A workspace that holds the rotated rows but not all the partial tiles the plan wants (a buffer sized for
    other rows): plain and gate/up calls run with what fits, against the oracle; one without room for the rows
    is refused."""
    k, n, K = 2048, 256, 3
    print(f"case: small workspace m={m}", flush=True)
    lib = _lib.lib()
    tg, su, sg = make_weight(k, n, K, seed=m)
    tu, _, sv_u = make_weight(k, n, K, seed=m + 1)
    sg, sv_u = ((v.astype(np.float32) * np.float32(4.0 / np.sqrt(k))).astype(np.float16) for v in (sg, sv_u))
    x = make_x(m, k, seed=m)
    xd, sud, tgd, sgd, tud, svd = (torch.from_numpy(v).cuda() for v in (x, su, tg, sg, tu, sv_u))
    base = (256 << 10) + (4 << 20) + m * k * 2 + ((m * (k // 128) * 4 + 255) & ~255)
    g = oracle.matmul(x, oracle.dequant(tg, su, sg, K, 1, rtz=True))
    u = oracle.matmul(x, oracle.dequant(tu, su, sv_u, K, 1, rtz=True))
    st = int(torch.cuda.current_stream().cuda_stream)
    assert base < lib.exl3_gemm_workspace_size(m, k, n, K) and base < lib.exl3_gate_up_workspace_size(m, k, n, K)
    for size in (base - 256, base, base + 2 * m * n * 4):
        ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
        y, z = (torch.zeros((m, n), dtype=torch.float16, device="cuda") for _ in range(2))
        rc = lib.exl3_gemm(xd.data_ptr(), tgd.data_ptr(), sud.data_ptr(), sgd.data_ptr(), y.data_ptr(), m, k, n, K, 1,
                           ws.data_ptr(), size, st)
        rc2 = lib.exl3_gate_up_swiglu(xd.data_ptr(), sud.data_ptr(), tgd.data_ptr(), sgd.data_ptr(), tud.data_ptr(),
                                      svd.data_ptr(), z.data_ptr(), m, k, n, K, 1, 0.0, ws.data_ptr(), size, st)
        if size < base:
            assert rc == rc2 == _lib.EXL3_ERR_WORKSPACE
            continue
        assert rc == rc2 == _lib.EXL3_OK
        check_close(y.float().cpu().numpy(), g, f"gemm m={m} in {size} bytes")
        check_close(z.float().cpu().numpy(), oracle.swiglu(g, u, float("inf")), f"gate/up m={m} in {size} bytes")


@pytest.mark.parametrize("kind", ["1", "1 whole", "128", "256"])
@pytest.mark.parametrize("m,k,n,K,cb,splits,limit", [
    (17, 128, 128, 1, 1, 1, 0.0), (31, 256, 384, 2, 2, 2, 1.0), (32, 512, 128, 3, 0, 4, 0.0),
    (33, 1024, 256, 4, 1, 8, 0.0), (127, 384, 128, 5, 2, 1, 2.0), (128, 256, 256, 6, 0, 2, 0.0),
    (129, 512, 384, 7, 1, 4, 0.0), (255, 128, 128, 8, 2, 1, 0.0), (256, 512, 256, 3, 2, 2, 0.0),
    (257, 256, 128, 4, 0, 1, 0.0), (520, 1024, 128, 3, 1, 1, 0.0)])
def test_gate_up_tall_tiles(m, k, n, K, cb, splits, limit, kind, monkeypatch):
    """gate/up + SwiGLU on tall tiles: partial tiles of either height with the finish launch, or both projections in
    one workgroup of up to 256 rows ("1 whole") or of a quarter of them ("1": these grids leave most CUs idle, so
    every tile runs as four row parts), at the edges of their row groups, every K and codebook: against the oracle,
    bit-equal when repeated and into an output that is only 4-byte aligned."""
    print(f"case: gate/up tall kind={kind} m={m} k={k} n={n} K={K} cb={cb} splits={splits}", flush=True)
    monkeypatch.setenv("EXL3_GU_TALL", kind.split()[0])
    if kind == "1 whole":
        monkeypatch.setenv("EXL3_FAT_TAIL", "0")
    monkeypatch.setenv("EXL3_FAT_SPLITS", str(splits))
    tg, su, sg = make_weight(k, n, K, seed=m + K)
    tu, _, sv_u = make_weight(k, n, K, seed=m + K + 50)
    scale = np.float32(4.0 / np.sqrt(k))
    sg, sv_u = ((v.astype(np.float32) * scale).astype(np.float16) for v in (sg, sv_u))
    x = make_x(m, k, seed=m)
    d = [torch.from_numpy(v).cuda() for v in (x, su, tg, sg, tu, sv_u)]
    y = torch.ops.sglang_exl3.exl3_gate_up_swiglu(*d, K, cb, limit)
    assert torch.equal(y, torch.ops.sglang_exl3.exl3_gate_up_swiglu(*d, K, cb, limit))
    g = oracle.matmul(x, oracle.dequant(tg, su, sg, K, cb, rtz=True))
    u = oracle.matmul(x, oracle.dequant(tu, su, sv_u, K, cb, rtz=True))
    check_close(y.float().cpu().numpy(), oracle.swiglu(g, u, limit or float("inf")), f"gate/up tall m={m}")
    lib = _lib.lib()
    need = lib.exl3_gate_up_workspace_size(m, k, n, K)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    odd = torch.zeros(m * n + 2, dtype=torch.float16, device="cuda")
    rc = lib.exl3_gate_up_swiglu(*[t.data_ptr() for t in d], odd.data_ptr() + 4, m, k, n, K, cb, limit, ws.data_ptr(),
                                 need, int(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "exl3_gate_up_swiglu")
    assert torch.equal(odd[2:].view(m, n), y)


@pytest.mark.parametrize("m,k,n,K,cb,limit", [(1300, 128, 7168, 3, 1, 0.0), (1300, 256, 7168, 2, 2, 1.0),
                                              (1100, 128, 8192, 4, 0, 0.0)])
def test_gate_up_fused_whole_tiles_and_parts(m, k, n, K, cb, limit, monkeypatch):
    """The fused gate/up kernel with a full round of whole tiles before the tail's (256 CUs: 336 tiles, the last 80 in
    two row parts each; 320 tiles, the last 64 in four) and a ragged last row tile: against the oracle, and the bits
    of whole tiles throughout (EXL3_FAT_TAIL=0)."""
    print(f"case: fused gate/up tail m={m} k={k} n={n} K={K} cb={cb}", flush=True)
    monkeypatch.setenv("EXL3_GU_TALL", "1")
    tg, su, sg = make_weight(k, n, K, seed=m + K)
    tu, _, sv_u = make_weight(k, n, K, seed=m + K + 50)
    scale = np.float32(4.0 / np.sqrt(k))
    sg, sv_u = ((v.astype(np.float32) * scale).astype(np.float16) for v in (sg, sv_u))
    x = make_x(m, k, seed=m)
    d = [torch.from_numpy(v).cuda() for v in (x, su, tg, sg, tu, sv_u)]
    y = torch.ops.sglang_exl3.exl3_gate_up_swiglu(*d, K, cb, limit)
    assert torch.equal(y, torch.ops.sglang_exl3.exl3_gate_up_swiglu(*d, K, cb, limit))
    g = oracle.matmul(x, oracle.dequant(tg, su, sg, K, cb, rtz=True))
    u = oracle.matmul(x, oracle.dequant(tu, su, sv_u, K, cb, rtz=True))
    check_close(y.float().cpu().numpy(), oracle.swiglu(g, u, limit or float("inf")), f"fused gate/up m={m}")
    monkeypatch.setenv("EXL3_FAT_TAIL", "0")
    assert torch.equal(y, torch.ops.sglang_exl3.exl3_gate_up_swiglu(*d, K, cb, limit))


@pytest.mark.parametrize("m,k,n,cb", [(16, 4096, 2048, 1), (64, 4096, 2048, 2), (14, 14336, 4608, 2),
                                      (16, 14336, 4608, 1)])
def test_gemm_split_handoff_repeatable(m, k, n, cb, monkeypatch):
    """exl3_gemm's narrow k-splits hand partial tiles to the last split of each
    (column block, row tile), in the kernel or (16 rows, up to four splits) in a
    finish launch: against the oracle, bit-identical over repeated calls (the
    counters reset themselves), and close to the fp32-atomic path
    (EXL3_FAT_HANDOFF=0).  k = 4096, n = 2048: four splits of 16 steps
    (EXL3_FAT_TALL=0, which tall tiles would take); k = 14336, n = 4608: eight of
    28, the hand-off that a default plan runs in the kernel."""
    K = 3
    if n <= 4096:
        monkeypatch.setenv("EXL3_FAT_TALL", "0")
    print(f"case: gemm split hand-off m={m} k={k} n={n} cb={cb}", flush=True)
    x = torch.from_numpy(make_x(m, k, seed=61 + m)).cuda()
    tr, su, sv = make_weight(k, n, K, seed=62)
    d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
    run = lambda: torch.ops.sglang_exl3.exl3_gemm(x, *d, K, cb == 1)
    outs = [run() for _ in range(3)]
    torch.cuda.synchronize()
    for o in outs[1:]:
        assert torch.equal(o, outs[0]), "split hand-off: repeated calls differ"
    ref = oracle.matmul(x.cpu().numpy(), oracle.dequant(tr, su, sv, K, cb, rtz=True))
    check_close(outs[0].float().cpu().numpy(), ref, f"split hand-off m={m}")
    monkeypatch.setenv("EXL3_FAT_HANDOFF", "0")
    atomic = run()
    torch.cuda.synchronize()
    check_close(outs[0].float().cpu().numpy(), atomic.float().cpu().numpy(), f"hand-off vs atomics m={m}")


@pytest.mark.parametrize("m,cb", [(6, 2), (9, 1), (13, 0), (16, 2)])
def test_gemm_split_out_finish_matches_in_kernel_handoff(m, cb, monkeypatch):
    """From 6 to 16 rows exl3_gemm's narrow k-splits store their partial tiles
    and a second launch (fat_split_finish_kernel) finishes every row; its sums
    and epilogue are the in-kernel hand-off's, so both give the same bits
    (EXL3_FAT_SPLIT_OUT=0 keeps the hand-off), mul1 raw entries included."""
    k, n, K = 2048, 384, 3
    print(f"case: gemm split-out finish m={m} cb={cb}", flush=True)
    monkeypatch.setenv("EXL3_GEMM_GEMV_ROWS", "0")  # the MFMA path at every m
    monkeypatch.setenv("EXL3_FAT_TALL", "0")  # 16-row tiles at 13 and 16 rows too
    x = torch.from_numpy(make_x(m, k, seed=81 + m)).cuda()
    tr, su, sv = make_weight(k, n, K, seed=82 + cb)
    d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
    run = lambda: torch.ops.sglang_exl3.exl3_linear(x, *d, K, cb)
    split = run()
    monkeypatch.setenv("EXL3_FAT_SPLIT_OUT", "0")
    handoff = run()
    torch.cuda.synchronize()
    assert torch.equal(split.view(torch.int16), handoff.view(torch.int16))
    ref = oracle.matmul(x.cpu().numpy(), oracle.dequant(tr, su, sv, K, cb, rtz=True))
    check_close(split.float().cpu().numpy(), ref, f"split-out m={m} cb={cb}")


@pytest.mark.parametrize("m", [13, 40, 100, 250])
@pytest.mark.parametrize("cb", [0, 1, 2])
def test_gemm_split_handoff_ragged_rows(m, cb, monkeypatch):
    """The split hand-off of the narrow kernel (EXL3_FAT_TALL=0) on row counts
    that leave the last row tile partial (16-row tiles at 13 rows, 64-row tiles
    above), every codebook (3INST through exl3_linear): k = 2048 gives two splits
    of 16 steps, n = 384 three column blocks.  Against the oracle, and
    bit-identical on a repeat call."""
    k, n, K = 2048, 384, 4
    monkeypatch.setenv("EXL3_FAT_TALL", "0")
    print(f"case: gemm split hand-off ragged m={m} cb={cb}", flush=True)
    x = torch.from_numpy(make_x(m, k, seed=71 + m)).cuda()
    tr, su, sv = make_weight(k, n, K, seed=72 + cb)
    d = [torch.from_numpy(v).cuda() for v in (tr, su, sv)]
    run = lambda: torch.ops.sglang_exl3.exl3_linear(x, *d, K, cb)
    first, again = run(), run()
    torch.cuda.synchronize()
    assert torch.equal(first, again), "split hand-off: repeated calls differ"
    ref = oracle.matmul(x.cpu().numpy(), oracle.dequant(tr, su, sv, K, cb, rtz=True))
    check_close(first.float().cpu().numpy(), ref, f"split hand-off ragged m={m} cb={cb}")


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
def test_fat_narrow_every_width(K, cb):
    """Narrow kernel (64-row tiles, fp32 output through exl3_fat_gemm) at every
    bit width and codebook: the decode's windows (middle words for the ones
    that straddle two words) differ per K."""
    M, k, n = 24, 512, 256
    print(f"case: fat narrow M={M} k={k} n={n} K={K} cb={cb}", flush=True)
    tr, su, sv = make_weight(k, n, K, seed=200 + 3 * K + cb)
    a = _rotate(make_x(M, k, seed=K + 20 * cb), su)
    check_close(_fat(a, tr, sv, K, cb, M, n), _ref(a, tr, sv, K, cb), f"fat narrow K={K} cb={cb}")


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", [1, 2])
def test_gemm_16_rows_every_width(K, cb, monkeypatch):
    """exl3_gemm at 16 rows (16-row tiles, which tall tiles replace at this width
    unless EXL3_FAT_TALL=0; mul1 reads raw entries) at every bit width, against
    the oracle."""
    m, k, n = 16, 1024, 256
    monkeypatch.setenv("EXL3_FAT_TALL", "0")
    print(f"case: gemm 16 rows K={K} cb={cb}", flush=True)
    tr, su, sv = make_weight(k, n, K, seed=300 + 3 * K + cb)
    x = make_x(m, k, seed=301 + K)
    d = [torch.from_numpy(v).cuda() for v in (x, tr, su, sv)]
    y = torch.ops.sglang_exl3.exl3_gemm(*d, K, cb == 1)
    torch.cuda.synchronize()
    ref = oracle.matmul(x, oracle.dequant(tr, su, sv, K, cb, rtz=True))
    check_close(y.float().cpu().numpy(), ref, f"gemm 16 rows K={K} cb={cb}")
