"""The native torch functions (csrc/sy_torch.cpp) against the Python autograd functions
they stand in for: the same bits, the same treatment of layouts, hooks and streams, and
every call that is not ordinary left to the Python path."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from switchyard import _lib, hip_op, stats_op, table_op  # noqa: E402
from switchyard.hip_op import block_attn_res_batched, block_attn_res_batched_train, block_attn_res_hip  # noqa: E402

DEV = "cuda"
EPS = 1e-6


def _make(n=9, b=2, t=33, d=512, s=None, dtype=torch.bfloat16, wdt=None, seed=0):
    g = torch.Generator().manual_seed(seed)
    v = torch.randn(n, b, t, d, generator=g).to(dtype).to(DEV)
    w = torch.randn(*((s, d) if s else (d,)), generator=g).mul(0.5).to(wdt or dtype).to(DEV)
    go = torch.randn(*((s,) if s else ()), b, t, d, generator=g).to(dtype).to(DEV)
    return v, w, go


# (name, public function, Python autograd function over (v, w), queries)
OPS = [
    ("op", lambda v, w: block_attn_res_hip(v, w, EPS), lambda v, w: hip_op._BlockAttnResHIP.apply(v, w, EPS), None),
    ("two_phase", lambda v, w: stats_op.block_attn_res_two_phase(v, w, 4, EPS),
     lambda v, w: stats_op._TwoPhase.apply(v, w, 4, EPS), None),
    ("batched", lambda v, w: block_attn_res_batched_train(v, w, EPS),
     lambda v, w: hip_op._BlockAttnResBatched.apply(v, w, EPS), 5),
    ("sources", lambda v, w: table_op.block_attn_res_sources(list(v.unbind(0)), w, EPS),
     lambda v, w: table_op._BlockAttnResSources.apply(w, EPS, *v.unbind(0)), None),
]


@pytest.mark.parametrize("op", OPS, ids=[o[0] for o in OPS])
@pytest.mark.parametrize("layout", ["dense", "strided", "misaligned"])
@pytest.mark.parametrize("wants", ["both", "v", "w"])
def test_native_equals_the_python_function(op, layout, wants):
    _, native, python, s = op
    v, w, go = _make(s=s)
    if layout == "strided":  # a transposed view, an expanded gradient
        v = v.transpose(1, 2).contiguous().transpose(1, 2)
        go = go[..., :1].expand_as(go)
    elif layout == "misaligned":  # rows one element past 16-byte alignment
        buf = torch.empty(v.numel() + 1, device=DEV, dtype=v.dtype)
        v = buf[1:].view_as(v).copy_(v)
    got = []
    for fn in (native, python):
        vv = v.detach().requires_grad_(wants != "w")
        ww = w.detach().requires_grad_(wants != "v")
        out = fn(vv, ww)
        leaves = [x for x in (vv, ww) if x.requires_grad]
        got.append([out.detach(), *torch.autograd.grad(out, leaves, go)])
    assert all(a.dtype == b.dtype and torch.equal(a, b) for a, b in zip(*got))
    with torch.no_grad():
        assert torch.equal(native(v, w), python(v, w)) and not native(v, w).requires_grad


def test_the_native_path_is_the_one_that_runs():
    v, w, _ = _make()
    q = _make(s=3)[1]
    m = _lib.native()
    assert m.block_attn_res(v, w, EPS) is not None and m.block_attn_res_batched(v, q, EPS) is not None
    assert m.block_attn_res_sources(list(v), w, EPS) is not None
    assert torch.equal(block_attn_res_batched(v, q), m.block_attn_res_batched(v, q, EPS))
    # left to Python: what its checks refuse or handle
    assert m.block_attn_res(v, w[:-1], EPS) is None and m.block_attn_res(v.cpu(), w.cpu(), EPS) is None
    assert m.block_attn_res(v[:, :, :0], w, EPS) is None and m.block_attn_res(v.double(), w, EPS) is None
    assert m.block_attn_res_two_phase(v, w, 9, EPS) is None
    assert m.block_attn_res_batched(v.requires_grad_(), q, EPS) is None


def test_saved_tensor_hooks_and_the_graph_rules():
    v, w, go = _make()
    v.requires_grad_()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.clone())[1], lambda t: t):
        out = block_attn_res_hip(v, w)
    assert v.shape in packed and w.shape in packed
    ref = torch.autograd.grad(block_attn_res_hip(v, w), v, go)[0]
    assert torch.equal(torch.autograd.grad(out, v, go)[0], ref)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, v, go)
    ww = w.clone()
    out = block_attn_res_hip(v, ww)
    ww.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, v, go)


def test_transforms_and_forward_mode_are_refused_as_before():
    v, w, _ = _make(b=1)
    with pytest.raises(RuntimeError, match="setup_context|functorch"):
        torch.func.vmap(lambda x: block_attn_res_hip(x, w))(torch.stack([v, v]))
    with pytest.raises(RuntimeError, match="setup_context|functorch"):
        torch.func.grad(lambda x: block_attn_res_hip(x, w).float().sum())(v)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(v, torch.ones_like(v))
        with pytest.raises((RuntimeError, NotImplementedError)):
            block_attn_res_hip(dual, w)


def test_another_stream_and_a_thread():
    import threading

    v, w, go = _make(t=300)
    v.requires_grad_()
    ref = torch.autograd.grad(block_attn_res_hip(v, w), v, go)[0]
    torch.cuda.synchronize()
    side, got = torch.cuda.Stream(), []

    def work():
        with torch.cuda.stream(side):
            got.append(torch.autograd.grad(block_attn_res_hip(v, w), v, go)[0])
        side.synchronize()

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert torch.equal(got[0], ref)
