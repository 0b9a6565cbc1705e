"""Infinities and NaN in one token, through every kernel that forms sums of more than one
row, chunk or query at once: that token is lost as the mathematics has it (an infinite
source has r = 0 and so a NaN logit), every other token keeps its bits, and only the
query gradients that it enters are lost with it."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from switchyard import _lib, hip_op  # noqa: E402
from switchyard.triton_op import BlockAttnResTriton, block_attn_res_triton  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32
POISON = [math.inf, -math.inf, math.nan]


def _rand(*shape, dtype, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def _run(call, v, leaves, go):
    vv = v.clone().requires_grad_()
    ll = [x.clone().requires_grad_() for x in leaves]
    out = call(vv, *ll)
    return [out.detach(), *torch.autograd.grad(out, [vv, *ll], go)]


# (name, N, T, D, dtype, query dtype): rows of any start, wide and two-factor queries in
# registers, in LDS, split and with the widest rows
OPS = [("op", 5, 9, 777, HF, HF), ("op", 12, 9, 1001, BF, F), ("op", 3, 5, 2050, F, F), ("op", 9, 40, 2048, BF, F),
       ("module", 9, 520, 4104, BF, BF), ("module", 9, 520, 4104, HF, HF), ("module", 4, 3, 8200, BF, BF),
       ("module", 16, 40, 1024, BF, F)]


@pytest.mark.parametrize("case", OPS)
@pytest.mark.parametrize("poison", POISON)
def test_one_token_of_the_operator(case, poison):
    kind, n, t, d, vdt, wdt = case
    print(f"nonfinite {case} {poison}", flush=True)
    v, go, w = _rand(n, 1, t, d, dtype=vdt, seed=1), _rand(1, t, d, dtype=vdt, seed=2), _rand(d, dtype=wdt, seed=3) * d**-0.5
    if kind == "op":
        call, leaves = (lambda v, w: block_attn_res_triton(v, w, 1e-6)), [w]
    else:
        mod = BlockAttnResTriton(d).to(DEV)
        call = lambda v, w, g: _lib.native().block_attn_res_gain(v, w, g, mod.eps)  # noqa: E731
        leaves = [w, 1 + 0.1 * _rand(d, dtype=wdt, seed=4)]
    clean = _run(call, v, leaves, go)
    tok, rest = t // 2, [k for k in range(t) if k != t // 2]
    for col in (0, d - 1, d - 7, d // 2):  # the last chunk of a row that is no whole chunks is read twice
        bad = v.clone()
        bad[n - 1, 0, tok, col] = poison
        out, dv, *dq = _run(call, bad, leaves, go)
        assert not out[0, tok].isfinite().any() and torch.equal(out[:, rest], clean[0][:, rest])
        assert not dv[:, 0, tok].isfinite().any() and torch.equal(dv[:, :, rest], clean[1][:, :, rest])
        assert not any(x.isfinite().any() for x in dq)
    bad = go.clone()
    bad[0, tok, d - 1] = poison
    out, dv, *dq = _run(call, v, leaves, bad)
    assert torch.equal(out, clean[0]) and torch.equal(dv[:, :, rest], clean[1][:, :, rest])
    assert not dv[:, 0, tok].isfinite().any() and not any(x.isfinite().any() for x in dq)


# any-row forward with two passes, with the element-wise backward, fp32, a wave per token
BATCHED = [(12, 8, 9, 1280, BF), (9, 5, 9, 777, HF), (12, 8, 9, 1028, F), (9, 8, 9, 4096, BF), (9, 8, 1100, 256, HF)]


@pytest.mark.parametrize("case", BATCHED)
@pytest.mark.parametrize("poison", POISON)
def test_one_token_of_the_batched_operator(case, poison):
    n, s, t, d, dt = case
    print(f"nonfinite batched {case} {poison}", flush=True)
    v, go, q = _rand(n, 1, t, d, dtype=dt, seed=1), _rand(s, 1, t, d, dtype=dt, seed=2), _rand(s, d, dtype=dt, seed=3) * d**-0.5
    call = lambda v, q: hip_op.block_attn_res_batched_train(v, q, 1e-6)  # noqa: E731
    clean = _run(call, v, [q], go)
    tok, rest = t // 2, [k for k in range(t) if k != t // 2]
    for col in (0, d - 1, d // 2):
        bad = v.clone()
        bad[n - 1, 0, tok, col] = poison
        out, dv, dq = _run(call, bad, [q], go)
        assert not out[:, 0, tok].isfinite().any() and torch.equal(out[:, :, rest], clean[0][:, :, rest])
        assert not dv[:, 0, tok].isfinite().any() and torch.equal(dv[:, :, rest], clean[1][:, :, rest])
        assert not dq.isfinite().any()
    bad = go.clone()
    bad[1, 0, tok, d - 1] = poison
    out, dv, dq = _run(call, v, [q], bad)
    assert torch.equal(out, clean[0]) and torch.equal(dv[:, :, rest], clean[1][:, :, rest])
    assert not dv[:, 0, tok].isfinite().any() and not dq[1].isfinite().any()
    others = [k for k in range(s) if k != 1]
    assert torch.equal(dq[others], clean[2][others])


@pytest.mark.parametrize("dtype", [BF, HF, F])
@pytest.mark.parametrize("poison", [*POISON, torch.finfo(torch.float16).max])
def test_sublayers_lose_what_the_plain_operations_lose(dtype, poison):
    print(f"nonfinite sublayers {dtype} {poison}", flush=True)
    m = _lib.native()
    x, w, g = _rand(5, 64, dtype=dtype, seed=1), _rand(64, dtype=dtype, seed=2), _rand(5, 64, dtype=dtype, seed=3)
    x[2, 5] = poison

    def norm(x, w):
        x, w = x.float(), w.float()
        return (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w).to(dtype)

    def swiglu(x):
        a, b = x.float().chunk(2, -1)
        return (torch.nn.functional.silu(a) * b).to(dtype)

    for fused, plain, leaves, go in ((lambda x, w: m.rms_norm(x, w, 1e-6), norm, [x, w], g),
                                     (m.swiglu, swiglu, [x], g[:, :32].contiguous())):
        got = _run(lambda a, *r: fused(a, *r), leaves[0], leaves[1:], go)
        ref = _run(lambda a, *r: plain(a, *r), leaves[0], leaves[1:], go)
        for a, b in zip(got, ref):
            assert torch.equal(a.isfinite(), b.isfinite()) and torch.equal(a.isnan(), b.isnan())
