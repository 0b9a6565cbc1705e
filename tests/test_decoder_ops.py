"""The decoder's fused sublayer kernels (RMSNorm, rotary with the QKV split, SwiGLU)
forward and backward against float64 torch, at rows of one chunk, partial lanes, the
widest row, one token and several per wave; and what is left to the plain operations."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle.reference import dtype_floor, rel_l2  # noqa: E402
from switchyard import _lib  # noqa: E402
from switchyard.model import Attention, ModelConfig, Rotary, Transformer  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32
DTYPES = [BF, HF, F]


def _rand(*shape, dtype, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def _close(got, ref, dtype):
    # one rounding of each output; fp32: sums of up to 4096 products
    assert rel_l2(got, ref.cpu()) <= (2e-6 if dtype == F else 1.10 * dtype_floor(ref.cpu(), dtype))


@pytest.mark.parametrize("shape", [(1, 8), (5, 64), (3, 520), (2, 7, 1032), (2100, 512), (33, 2048), (9, 4096)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_rms_norm(shape, dtype):
    d = shape[-1] // 2 if dtype == F else shape[-1]
    shape = (*shape[:-1], d)
    x, w, g = _rand(*shape, dtype=dtype, seed=1), _rand(d, dtype=dtype, seed=2), _rand(*shape, dtype=dtype, seed=3)
    xx, ww = x.clone().requires_grad_(), w.clone().requires_grad_()
    out = _lib.native().rms_norm(xx, ww, 1e-6)
    dx, dw = torch.autograd.grad(out, (xx, ww), g)
    x6, w6 = x.double().requires_grad_(), w.double().requires_grad_()
    ref = x6 * torch.rsqrt(x6.square().mean(-1, keepdim=True) + 1e-6) * w6
    rdx, rdw = torch.autograd.grad(ref, (x6, w6), g.double())
    for got, want in ((out.detach(), ref.detach()), (dx, rdx), (dw, rdw)):
        assert got.dtype == dtype and got.shape == want.shape
        _close(got, want, dtype)
    with torch.no_grad():
        assert torch.equal(_lib.native().rms_norm(x, w, 1e-6), out)


@pytest.mark.parametrize("bthd", [(1, 1, 1, 16), (2, 33, 3, 64), (3, 7, 2, 48), (1, 300, 4, 128)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_rope_qkv(bthd, dtype):
    b, t, h, hd = bthd
    rot = Rotary(hd, 512, 10000.0).to(DEV)
    qkv = _rand(b, t, 3, h, hd, dtype=dtype, seed=4)
    gs = [_rand(b, h, t, hd, dtype=dtype, seed=5 + k) for k in range(3)]
    gs[1] = gs[1].transpose(1, 2).contiguous().transpose(1, 2)  # a strided gradient
    xx = qkv.clone().requires_grad_()
    out = _lib.native().rope_qkv(xx, rot.cos, rot.sin)
    dq = torch.autograd.grad(out, xx, gs)[0]
    x6 = qkv.double().requires_grad_()
    cos, sin = rot.cos[:t].double(), rot.sin[:t].double()

    def turn(x):
        lo, hi = x.chunk(2, -1)
        return torch.cat((lo * cos - hi * sin, lo * sin + hi * cos), -1)

    q, k, v = x6.unbind(2)
    ref = [y.transpose(1, 2) for y in (turn(q), turn(k), v)]
    rdq = torch.autograd.grad(ref, x6, [g.double() for g in gs])[0]
    for got, want in (*zip(out, ref), (dq, rdq)):
        assert got.is_contiguous() and got.shape == want.shape
        _close(got.detach(), want.detach(), dtype)


@pytest.mark.parametrize("shape", [(1, 16), (3, 5, 2816), (700, 208)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_swiglu(shape, dtype):
    x = _rand(*shape, dtype=dtype, seed=8) * 3
    x[0, ..., 0] = 90.0  # saturated gates
    x[0, ..., 1] = -90.0
    g = _rand(*shape[:-1], shape[-1] // 2, dtype=dtype, seed=9)
    xx = x.clone().requires_grad_()
    out = _lib.native().swiglu(xx)
    dx = torch.autograd.grad(out, xx, g)[0]
    x6 = x.double().requires_grad_()
    a, u = x6.chunk(2, -1)
    ref = torch.nn.functional.silu(a) * u
    _close(out.detach(), ref.detach(), dtype)
    _close(dx, torch.autograd.grad(ref, x6, g.double())[0], dtype)


@pytest.mark.parametrize("op", ["rms_norm", "frozen_norm", "swiglu", "rope_qkv"])
def test_second_derivatives(op):
    """A recorded backward (create_graph) can itself be differentiated, as through the
    plain operations; fp32 sums of at most 64 products and their products: 1e-5."""
    print(f"second derivatives {op}", flush=True)
    m = _lib.native()
    rot = Rotary(16, 8, 1e4).to(DEV)
    shape = (2, 8, 3, 2, 16) if op == "rope_qkv" else (5, 64)
    x, w = _rand(*shape, dtype=F, seed=1), _rand(64, dtype=F, seed=2)

    def call(x, w):
        if op in ("rms_norm", "frozen_norm"):
            return [m.rms_norm(x, w, 1e-6)] if x.dtype == F else [x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w]
        if op == "swiglu":
            a, u = x.chunk(2, -1)
            return [m.swiglu(x)] if x.dtype == F else [torch.nn.functional.silu(a) * u]
        if x.dtype == F:
            return m.rope_qkv(x, rot.cos, rot.sin)
        lo, hi = x[:, :, :2].chunk(2, -1)
        c, s = (y[:8].reshape(8, 1, 1, 8).double() for y in (rot.cos, rot.sin))
        qk = torch.cat((lo * c - hi * s, lo * s + hi * c), -1)
        return [y.transpose(1, 2) for y in (*qk.unbind(2), x[:, :, 2])]

    got = []
    for dtype in (F, torch.float64):
        xx, ww = x.to(dtype).requires_grad_(), w.to(dtype).requires_grad_(op != "frozen_norm")
        leaves = [xx, ww] if op == "rms_norm" else [xx]
        first = torch.autograd.grad(sum(y.pow(3).sum() for y in call(xx, ww)), leaves, create_graph=True)
        got.append([*first, *torch.autograd.grad(sum(y.square().sum() for y in first), leaves)])
    for a, b in zip(*got):
        assert rel_l2(a.detach().cpu(), b.detach().cpu()) <= 1e-5


def test_other_tensors_are_left_to_the_plain_operations():
    m = _lib.native()
    x, w = _rand(4, 64, dtype=BF, seed=1), _rand(64, dtype=BF, seed=2)
    assert m.rms_norm(x, w.float(), 1e-6) is None and m.rms_norm(x.t(), w[:4], 1e-6) is None
    assert m.rms_norm(x[:, :63], w[:63], 1e-6) is None and m.rms_norm(x.cpu(), w.cpu(), 1e-6) is None
    assert m.swiglu(x[:, ::2]) is None and m.swiglu(x[:, :24].contiguous()) is None
    rot = Rotary(16, 8, 1e4).to(DEV)
    qkv = _rand(1, 9, 3, 2, 16, dtype=BF, seed=3)  # more positions than the tables hold
    assert m.rope_qkv(qkv, rot.cos, rot.sin) is None
    assert m.rope_qkv(qkv[:, :8], rot.cos.double(), rot.sin) is None


@pytest.mark.parametrize("residual", ["standard", "switchyard"])
def test_the_decoder_agrees_with_its_plain_operations(residual, monkeypatch):
    """Loss and gradients of a small fp32 decoder with the kernels and without."""
    cfg = ModelConfig(vocab_size=128, d_model=64, n_heads=2, d_ff=128, n_layers=2, n_blocks=2, max_seq_len=32,
                      residual=residual)
    torch.manual_seed(0)
    model = Transformer(cfg).to(DEV)
    if model.attn_res is not None:
        for site in model.attn_res:
            torch.nn.init.normal_(site.w, std=0.3)
    idx = torch.randint(0, 128, (2, 32), generator=torch.Generator().manual_seed(1)).to(DEV)
    got = []
    for plain in (False, True):
        if plain:
            monkeypatch.setattr(_lib, "ordinary", lambda *t: False)
        loss = model(idx, idx)[1]
        got.append([loss.detach(), *torch.autograd.grad(loss, list(model.parameters()))])
        with torch.no_grad():
            got[-1].append(model(idx))
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=2e-4, atol=2e-5)  # fp32 sums in another order, two layers deep


class _Turned(Rotary):
    def forward(self, x):
        return super().forward(x) * 2


def test_attention_calls_a_rotary_that_is_more_than_its_tables():
    """Hooks, a subclass, a replaced forward and tables that broadcast otherwise all act
    as they do on the plain operations; the plain rotary's kernel agrees with them."""
    torch.manual_seed(0)
    cfg = ModelConfig(vocab_size=128, d_model=64, n_heads=2, d_ff=128, n_layers=2, n_blocks=2, max_seq_len=32)
    attn, rot, x = Attention(cfg).to(DEV), Rotary(32, 32, 1e4).to(DEV), _rand(2, 8, 64, dtype=F, seed=1)
    ref, calls = attn(x, rot), []
    hook = rot.register_forward_hook(lambda *a: calls.append(1))
    torch.testing.assert_close(attn(x, rot), ref)
    hook.remove()
    assert len(calls) == 2
    hook = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: calls.append(1) if m is rot else None)
    attn(x, rot)
    hook.remove()
    assert len(calls) == 4
    sub = _Turned(32, 32, 1e4).to(DEV)
    replaced = Rotary(32, 32, 1e4).to(DEV)
    replaced.forward = lambda y: Rotary.forward(replaced, y) * 2
    torch.testing.assert_close(attn(x, sub), attn(x, replaced))
    assert not torch.allclose(attn(x, sub), ref)
    with torch.no_grad():
        assert torch.equal(attn(x, rot), ref) and not calls[4:]
    # positions along the batch, as broadcasting has it: refused by the plain operations
    rot.cos, rot.sin = rot.cos[:, 0], rot.sin[:, 0]
    with pytest.raises(RuntimeError):
        attn(x, rot)


def _sublayer(op):
    """(function of the sublayer's inputs, inputs, the same from plain operations)."""
    m = _lib.native()
    if op == "rms_norm":
        leaves = [_rand(5, 64, dtype=F, seed=1), _rand(64, dtype=F, seed=2)]
        return (lambda x, w: m.rms_norm(x, w, 1e-6)), leaves, lambda x, w: (
            x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w)
    if op == "swiglu":
        return m.swiglu, [_rand(5, 64, dtype=F, seed=1)], lambda x: torch.nn.functional.silu(x[:, :32]) * x[:, 32:]
    rot = Rotary(16, 8, 1e4).to(DEV)

    def plain(x):
        q, k, v = x.unbind(2)
        return torch.stack([y.transpose(1, 2) for y in (rot(q), rot(k), v)])

    return (lambda x: torch.stack(m.rope_qkv(x, rot.cos, rot.sin))), [_rand(2, 8, 3, 2, 16, dtype=F, seed=1)], plain


@pytest.mark.parametrize("op", ["rms_norm", "swiglu", "rope_qkv"])
def test_a_backward_inside_a_transform_or_mode(op):
    """Ordinary forwards whose backward is not: batched gradients, a dispatch mode, a
    gradient with a tangent. fp32 sums of at most 64 products on both sides: 1e-5."""
    print(f"backward inside a transform {op}", flush=True)
    fused, leaves, plain = _sublayer(op)
    leaves = [x.requires_grad_() for x in leaves]
    out, ref = fused(*leaves), plain(*leaves)
    g = _rand(3, *out.shape, dtype=F, seed=5)
    got = torch.autograd.grad(out, leaves, g, is_grads_batched=True, retain_graph=True)
    for k in range(3):
        want = torch.autograd.grad(ref, leaves, g[k], retain_graph=True)
        for a, b in zip(got, want):
            assert rel_l2(a[k].cpu(), b.cpu()) <= 1e-5
    jac = torch.autograd.functional.jacobian(lambda x: fused(x, *leaves[1:])[:1].flatten()[:4], leaves[0], vectorize=True)
    assert jac.shape == (4, *leaves[0].shape)

    class Seen(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    seen = []
    with Seen():
        got = torch.autograd.grad(out, leaves, g[0], retain_graph=True)
    assert any("mul" in str(f) for f in seen)
    for a, b in zip(got, torch.autograd.grad(ref, leaves, g[0], retain_graph=True)):
        assert rel_l2(a.cpu(), b.cpu()) <= 1e-5
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(g[0].clone(), g[1])
        got = torch.autograd.grad(out, leaves, dual, retain_graph=True)
        tangent = torch.autograd.forward_ad.unpack_dual(got[0]).tangent
    want = torch.autograd.grad(ref, leaves, g[1])[0]  # the gradient is linear in g
    assert rel_l2(tangent.cpu(), want.cpu()) <= 1e-5


@pytest.mark.parametrize("dtype", [BF, F])
def test_the_sites_agree_bit_for_bit_in_every_mode(dtype):
    """Trained queries (no zeros, no unit gains): the three ways of presenting sources,
    with and without a backward to come, see the same query and give the same bits."""
    print(f"site bits {dtype}", flush=True)
    outs = {}
    for sources in ("stack", "arena", "table"):
        torch.manual_seed(0)
        cfg = ModelConfig(vocab_size=128, d_model=128, n_heads=2, d_ff=128, n_layers=3, n_blocks=3, max_seq_len=32,
                          residual="switchyard", sources=sources)
        model = Transformer(cfg)
        for site in model.attn_res:
            torch.nn.init.normal_(site.w, std=0.3)
            torch.nn.init.normal_(site.g, mean=1.0, std=0.3)
        model = model.to(DEV, dtype)
        idx = torch.randint(0, 128, (2, 32), generator=torch.Generator().manual_seed(1)).to(DEV)
        outs[sources, True] = model(idx).detach()
        with torch.no_grad():
            outs[sources, False] = model(idx)
            assert torch.equal(model(idx, collect_alphas=True), outs[sources, False])
    ref = outs["stack", True]
    assert all(torch.equal(x, ref) for x in outs.values())


def test_a_norm_over_more_tokens_than_one_launch_has_waves():
    """2^26 tokens of a wave each would be 2^32 threads, which is no launch."""
    t = (1 << 26) + 5
    print("rms_norm at 2^26 tokens", flush=True)
    x = torch.zeros(t, 8, device=DEV, dtype=BF)
    rows = torch.tensor([0, 1, (1 << 22) + 3, (1 << 26) - 1, t - 1], device=DEV)
    x[rows] = _rand(5, 8, dtype=BF, seed=1)
    w, g = _rand(8, dtype=BF, seed=2), _rand(5, 8, dtype=BF, seed=3)
    go = torch.zeros_like(x)
    go[rows] = g
    small = [y.clone().requires_grad_() for y in (x[rows], w)]
    big = [x.requires_grad_(), w.clone().requires_grad_()]
    want = torch.autograd.grad(_lib.native().rms_norm(*small, 1e-6), small, g)
    out = _lib.native().rms_norm(*big, 1e-6)
    dx, dw = torch.autograd.grad(out, big, go)
    assert torch.equal(out[rows], _lib.native().rms_norm(*small, 1e-6))
    assert torch.equal(dx[rows], want[0]) and rel_l2(dw.cpu(), want[1].double().cpu()) <= 4e-3  # one rounding
