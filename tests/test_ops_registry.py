"""torch.ops.sglang_exl3 registry and fake-tensor shape inference (CPU).

Mirrors the reference's tests/test_cuda_graph.py:13-68 (same op list, same fake
shapes), and checks that CPU tensors are refused (no CPU fallback)."""

import importlib.metadata
import os
import subprocess
import sys

import pytest
import torch

import sglang_exl3
from sglang_exl3 import ops

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang-exl3_amd")


@pytest.fixture(scope="module", autouse=True)
def _registered():
    sglang_exl3.register()
    ops.register_custom_ops()


def test_ops_registered_in_torch():
    for name in ops.OP_NAMES:
        assert hasattr(torch.ops.sglang_exl3, name), name


def test_meta_fake_tensor_dispatch():
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        x = torch.empty((2, 128), dtype=torch.float16)
        trellis = torch.empty((8, 16, 32), dtype=torch.int16)
        suh = torch.empty((128,), dtype=torch.float16)
        svh = torch.empty((256,), dtype=torch.float16)
        g = torch.ops.sglang_exl3.exl3_gemv(x, trellis, suh, svh, 2, True, 1)
        assert g.shape == (2, 256) and g.dtype == torch.float16
        gm = torch.ops.sglang_exl3.exl3_gemm(x, trellis, suh, svh, 2, True)
        assert gm.shape == (2, 256) and gm.dtype == torch.float16
        d = torch.ops.sglang_exl3.dequant_trellis(trellis, suh, svh, 2, True)
        assert d.shape == (128, 256) and d.dtype == torch.float16
        ptrs = torch.empty((4,), dtype=torch.int64)
        ids = torch.empty((6,), dtype=torch.int32)
        b = torch.ops.sglang_exl3.p2b_gemv_batched(x, ptrs, ptrs, ptrs, ids, 2, True, 768)
        assert b.shape == (6, 2, 768)
        b2 = torch.ops.sglang_exl3.p2b_gemv_batched(x, ptrs, ptrs, ptrs, ids, 2, True, 0)
        assert b2.shape == (6, 2, 2048)
        out = torch.empty((1, 128), dtype=torch.float16)
        w = torch.empty((6,), dtype=torch.float16)
        assert torch.ops.sglang_exl3.p2b_fused_moe(x[:1], out, ptrs, ptrs, ptrs, ptrs, ptrs, ptrs, ptrs, ptrs,
                                                   ptrs, ids, w, 2, 2, 2, True) is None
        xb = torch.empty((2, 128), dtype=torch.bfloat16)
        c = torch.ops.sglang_exl3.exl3_linear_cat(xb, [trellis, trellis], [suh, suh], [svh, svh], 2, 1, False)
        assert c.shape == (2, 512) and c.dtype == torch.float16
        c = torch.ops.sglang_exl3.exl3_linear_part(xb, [trellis] * 3, [suh] * 3, [svh] * 3, 2, 1, True, 1)
        assert c.shape == (1024,) and c.dtype == torch.bfloat16
        mo = torch.ops.sglang_exl3.exl3_moe_layer_typed(xb, ids, w, *[ptrs] * 9, 2, 2, 2, True, 128)
        assert mo.shape == (2, 128) and mo.dtype == torch.bfloat16
        o32 = torch.empty((2, 256), dtype=torch.float32)
        assert torch.ops.sglang_exl3.exl3_fat_gemm(x, trellis, o32, svh, 2, True, False) is None


@pytest.mark.parametrize("fault", ["missing", "other torch", "does not load"])
def test_operators_register_without_the_native_path(fault, tmp_path):
    """Without the second library, with one built for another PyTorch or one that does not load, the operators are
    registered all the same and keep their Python implementation."""
    lib = tmp_path / "libsglang_exl3_ops.so"
    if fault != "missing":
        version = importlib.metadata.version("torch") if fault == "does not load" else "0.0.1"
        lib.write_bytes(b"not a library exl3-ops-torch:" + version.encode() + b"\0")
    code = f"""
import sys
sys.path.insert(0, {PKG!r})
import torch
from sglang_exl3 import _lib, ops
_lib.OPS_LIB_PATH = {str(lib)!r}
assert ops.register_custom_ops() and not ops._NATIVE_PATH
x = torch.empty((2, 128), dtype=torch.float16, device="meta")
t, h = (torch.empty(s, dtype=d, device="meta") for s, d in (((8, 16, 32), torch.int16), ((256,), torch.float16)))
assert torch.ops.sglang_exl3.exl3_linear_cat(x, [t], [h], [h], 2, 1, False).shape == (2, 256)
try:
    torch.ops.sglang_exl3.exl3_gemv(torch.zeros((1, 128)), torch.zeros((8, 16, 32)), torch.zeros(128), torch.zeros(256), 2, True)
except RuntimeError as e:
    assert "HIP device" in str(e)
else:
    raise AssertionError
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.parametrize("fault", ["no compiler", "does not compile"])
def test_build_without_the_native_path(fault, tmp_path, monkeypatch, capsys):
    """Where the second library cannot be built, the build warns and leaves none behind that is out of date."""
    monkeypatch.syspath_prepend(PKG)
    import build_hip

    old = tmp_path / build_hip.OPS_LIBNAME
    old.write_bytes(b"an older one")
    (tmp_path / "torch_ops.cpp").write_text("#error")
    monkeypatch.setattr(build_hip, "LIBDIR", str(tmp_path))
    monkeypatch.setattr(build_hip, "CSRC", str(tmp_path))
    if fault == "no compiler":
        monkeypatch.setenv("PATH", str(tmp_path))
    build_hip._build_ops(force=False)
    assert "native entry is not built" in capsys.readouterr().err and not old.exists()


def test_cpu_tensors_are_refused():
    x = torch.zeros((1, 128), dtype=torch.float16)
    trellis = torch.zeros((8, 16, 32), dtype=torch.int16)
    suh = torch.ones(128, dtype=torch.float16)
    svh = torch.ones(256, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="HIP device"):
        torch.ops.sglang_exl3.exl3_gemv(x, trellis, suh, svh, 2, True, 1)
    with pytest.raises(RuntimeError, match="HIP device"):
        torch.ops.sglang_exl3.dequant_trellis(trellis, suh, svh, 2, True)
