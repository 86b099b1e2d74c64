"""The native path of the eager operators against their *_general twins (the Python path): the same bits for
the calls it takes, and the general path's results and errors for those it hands on."""

import threading

import pytest
import torch

from gpu_util import make_weight, make_x
from sglang_exl3 import ops

pytestmark = pytest.mark.gpu
K, k, n = 3, 256, 384


@pytest.fixture(scope="module", autouse=True)
def _registered():
    ops.register_custom_ops()


@pytest.fixture(scope="module")
def weights():
    return [[torch.from_numpy(a).cuda() for a in make_weight(k, n, K, seed=s)] for s in (1, 2, 3)]


def _calls(w, x):
    o = torch.ops.sglang_exl3
    tr, su, sv = ([t[j] for t in w] for j in range(3))
    return {
        "gemv": (o.exl3_gemv, o.exl3_gemv_general, (x, *w[0], K, True, 1)),
        "cat": (o.exl3_linear_cat, o.exl3_linear_cat_general, (x, tr, su, sv, K, 1, True)),
        "part": (o.exl3_linear_part, o.exl3_linear_part_general, (x, tr, su, sv, K, 2, False, 1)),
        "cat1": (o.exl3_linear_cat, o.exl3_linear_cat_general, (x.bfloat16(), tr[:1], su[:1], sv[:1], K, 2, False)),
        "gate_up": (o.exl3_gate_up_swiglu, o.exl3_gate_up_swiglu_general, (x, su[0], tr[0], sv[0], tr[1], sv[1], K, 1, 2.0)),
    }


def _same(op, general, args):
    outs = []
    for f in (general, op):
        try:
            outs.append(f(*args))
        except RuntimeError as e:
            outs.append((type(e), str(e)))
    assert torch.equal(*outs) if isinstance(outs[0], torch.Tensor) else outs[0] == outs[1]


@pytest.mark.parametrize("name", ["gemv", "cat", "part", "cat1", "gate_up"])
@pytest.mark.parametrize("m", [1, 17, 64])
def test_native_equals_general(weights, name, m, monkeypatch):
    print(f"case: native op {name} m={m}", flush=True)
    x = torch.from_numpy(make_x(m, k, seed=m)).cuda()
    op, general, args = _calls(weights, x)[name]
    want = general(*args)
    with monkeypatch.context() as mp:  # the Python implementation is not reached: the call is the native path's
        for impl in ("exl3_gemv_impl", "exl3_linear_cat_impl", "exl3_linear_part_impl", "exl3_gate_up_swiglu_impl"):
            mp.setattr(ops, impl, lambda *a: pytest.fail("general path"))
        for _ in range(2):
            got = op(*args)
            assert got.dtype == want.dtype and torch.equal(got, want)
    with torch.inference_mode():
        assert torch.equal(op(*args), want)
    # strided rows, three-dimensional rows, rows at an odd element offset
    wide = torch.zeros((m, 2 * k), dtype=args[0].dtype, device="cuda")
    wide[:, :k] = args[0]
    odd = torch.zeros(m * k + 1, dtype=args[0].dtype, device="cuda")
    odd[1:] = args[0].reshape(-1)
    for xs in (wide[:, :k], args[0].view(1, m, k), odd[1:].view(m, k)):
        _same(op, general, (xs, *args[1:]))
    # another stream (its own workspace), from another thread
    res = []

    def run():
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            res.extend(op(*args) for _ in range(2))
        s.synchronize()

    torch.cuda.synchronize()
    t = threading.Thread(target=run)
    t.start()
    t.join()
    assert len(res) == 2 and all(torch.equal(r, want) for r in res)


def test_native_refuses_what_general_refuses(weights):
    x = torch.from_numpy(make_x(2, k, seed=5)).cuda()
    for name, (op, general, args) in _calls(weights, x).items():
        for bad in ((x[:, :128], *args[1:]), (x.float(), *args[1:]), (x[0], *args[1:]), (x.cpu(), *args[1:])):
            _same(op, general, bad)
        empty = op(x[:0], *args[1:]) if name in ("cat", "part", "cat1", "gate_up") else None
        assert empty is None or empty.shape == general(x[:0], *args[1:]).shape
        xg = args[0].detach().clone().requires_grad_()
        y = op(xg, *args[1:])
        assert y.requires_grad and torch.equal(y.detach(), general(*args))
        with pytest.raises(RuntimeError):
            y.float().sum().backward()
