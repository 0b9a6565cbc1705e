"""The module's query as two factors, multiplied in the kernels: outputs and the
gradients of both factors on every family a two-factor query takes, against the
float64 oracle of the product."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle.reference import block_attn_res_oracle, dtype_floor, oracle_grads, rel_l2  # noqa: E402
from switchyard import _lib  # noqa: E402
from switchyard.triton_op import BlockAttnResTriton  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32

# (N, T, D): resident, chunked and tall tiles, the eight-wave row (element-wise
# backward), unaligned rows, and rows under 16 bytes (element-wise both ways)
SHAPES = [(9, 1100, 2048), (4, 3, 64), (16, 40, 1024), (32, 24, 2048), (3, 8, 16384), (5, 70, 777), (4, 20, 7)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtypes", [(BF, BF), (BF, F), (HF, HF), (F, F)])
@pytest.mark.parametrize("wants", ["all", "w"])
def test_module_with_a_gain(shape, dtypes, wants):
    vdt, wdt = dtypes
    n, t, d = shape
    print(f"gain {shape} {dtypes}", flush=True)
    g = torch.Generator().manual_seed(d)
    v = torch.randn(n, 1, t, d, generator=g).to(vdt)
    w = (torch.randn(d, generator=g) * d**-0.5).to(wdt)
    gain = (1 + 0.3 * torch.randn(d, generator=g)).to(wdt)
    go = torch.randn(1, t, d, generator=g).to(vdt)
    mod = BlockAttnResTriton(d).to(DEV).to(wdt)
    with torch.no_grad():
        mod.w.copy_(w)
        mod.g.copy_(gain)
    vv = v.to(DEV).requires_grad_(wants == "all")
    mod.g.requires_grad_(wants == "all")
    out = mod(vv)
    leaves = [x for x in (vv, mod.w, mod.g) if x.requires_grad]
    grads = torch.autograd.grad(out, leaves, go.to(DEV))
    q = w.double() * gain.double()
    rdv, rdq = oracle_grads(v.double(), q, go.double())
    ref = {id(vv): (rdv, vdt), id(mod.w): (rdq * gain.double(), wdt), id(mod.g): (rdq * w.double(), wdt)}
    for got, (want, dt) in ((out.detach(), (block_attn_res_oracle(v.double(), q), vdt)),
                            *((x, ref[id(leaf)]) for x, leaf in zip(grads, leaves))):
        assert got.dtype == dt
        assert rel_l2(got, want) <= (1e-5 if dt == F else 1.10 * dtype_floor(want, dt))
    with torch.no_grad():
        assert torch.equal(mod(vv), out)


@pytest.mark.parametrize("wdt", [BF, F])
def test_a_recorded_backward_can_be_differentiated_by_the_factors(wdt):
    """The operator's gradients carry no graph, the product's do: dw = dq g, dg = dq w."""
    n, t, d = 4, 40, 256
    gen = torch.Generator().manual_seed(3)
    v, go = torch.randn(n, 1, t, d, generator=gen).to(BF).to(DEV), torch.randn(1, t, d, generator=gen).to(BF).to(DEV)
    mod = BlockAttnResTriton(d).to(DEV).to(wdt)
    with torch.no_grad():
        mod.w.copy_(torch.randn(d, generator=gen) * d**-0.5)
        mod.g.copy_(1 + 0.3 * torch.randn(d, generator=gen))
    leaves = [mod.w, mod.g]
    plain = torch.autograd.grad(mod(v), leaves, go)
    dw, dg = torch.autograd.grad(mod(v), leaves, go, create_graph=True)
    for a, b in zip((dw, dg), plain):  # one rounding each of sums in the same order
        assert rel_l2(a.detach(), b.cpu().double()) <= (1e-6 if wdt == F else 4e-3)
    ww, gg = torch.autograd.grad((dw.float().sum() + 2 * dg.float().sum()), leaves)
    with torch.no_grad():
        dq = dg.double() / mod.w.double()
    for got, want in ((gg, dq), (ww, 2 * dq)):  # dg's rounding, and one of the result
        assert got.dtype == wdt and rel_l2(got, want.cpu()) <= (1e-5 if wdt == F else 1e-2)


# Nine-row four-chunk tiles on two, four and eight waves (past the tile rule for few
# tokens), at full rows and where the last chunks are partial, above and at one token.
LDS_SHAPES = [(9, 600, 4096), (7, 530, 2312), (9, 520, 8192), (5, 515, 4104), (9, 3, 16384), (6, 1, 8200)]


@pytest.mark.parametrize("shape", LDS_SHAPES)
@pytest.mark.parametrize("dtypes", [(BF, BF), (HF, HF), (BF, F), (HF, BF)])
def test_queries_held_in_lds(shape, dtypes):
    """The forward's factors in LDS: fp32 values, or a bf16 product in two exact parts. The
    logits themselves (the operator's stats) are within fp32 rounding of the exact
    product's: sums of up to D terms, at most 64 to a lane."""
    vdt, wdt = dtypes
    n, t, d = shape
    print(f"lds query {shape} {dtypes}", flush=True)
    gen = torch.Generator().manual_seed(d + t)
    v = torch.randn(n, 1, t, d, generator=gen).to(vdt)
    w = (torch.randn(d, generator=gen) * d**-0.5).to(wdt)
    gain = (1 + 0.3 * torch.randn(d, generator=gen)).to(wdt)
    vd, wd, gd = v.to(DEV), w.to(DEV), gain.to(DEV)
    out, stats = torch.empty(1, t, d, device=DEV, dtype=vdt), torch.empty(2, n, t, device=DEV)
    _lib.check(_lib.lib().sy_fwd_gain(vd.data_ptr(), wd.data_ptr(), gd.data_ptr(), out.data_ptr(), stats.data_ptr(),
                                      n, t, d, t * d, _lib.dtype_code(vdt), _lib.dtype_code(wdt), 1e-6,
                                      _lib.stream_ptr(vd.device)), "sy_fwd_gain")
    q = w.double() * gain.double()
    ref = block_attn_res_oracle(v.double(), q)
    assert rel_l2(out, ref) <= 1.10 * dtype_floor(ref, vdt)
    r = torch.rsqrt(v.double().square().mean(-1) + 1e-6)[:, 0]
    logits = (v.double() @ q)[:, 0] * r
    assert rel_l2(stats[0], logits) <= 2e-6 and rel_l2(stats[1], r) <= 1e-6


@pytest.mark.parametrize("shape", [(9, 300, 8200), (4, 270, 16384), (5, 2, 12288), (2, 300, 8200)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_gradients_of_the_widest_rows(shape, dtype):
    """The eight-wave tile with the factors in LDS: one and two tokens a workgroup, partial
    last chunks. Held to the floor of one rounding, which a rounded product does not meet."""
    n, t, d = shape
    print(f"widest rows {shape} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(d + t)
    v = torch.randn(n, 1, t, d, generator=gen).to(dtype)
    w = (torch.randn(d, generator=gen) * d**-0.5).to(dtype)
    gain = (1 + 0.3 * torch.randn(d, generator=gen)).to(dtype)
    go = torch.randn(1, t, d, generator=gen).to(dtype)
    mod = BlockAttnResTriton(d).to(DEV).to(dtype)
    with torch.no_grad():
        mod.w.copy_(w)
        mod.g.copy_(gain)
    vv = v.to(DEV).requires_grad_()
    dv, dw, dg = torch.autograd.grad(mod(vv), [vv, mod.w, mod.g], go.to(DEV))
    rdv, rdq = oracle_grads(v.double(), w.double() * gain.double(), go.double())
    for got, want in ((dv, rdv), (dw, rdq * gain.double()), (dg, rdq * w.double())):
        assert rel_l2(got, want) <= 1.10 * dtype_floor(want, dtype)


@pytest.mark.parametrize("size", [1e-7, 1e-4, 1.0, 250.0])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_split_products_of_any_size(size, dtype):
    """A lane's products from below fp16's normal range to beyond its largest number, of
    very different sizes within a lane: the logits keep fp32 accuracy."""
    n, t, d = 6, 515, 2312
    print(f"split products {size} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(7)
    v = torch.randn(n, 1, t, d, generator=gen).to(dtype)
    spread = torch.exp2(-torch.randint(0, 12, (d,), generator=gen).float())
    w, gain = (torch.randn(d, generator=gen) * size).to(dtype), (torch.randn(d, generator=gen) * size * spread).to(dtype)
    vd, wd, gd = v.to(DEV), w.to(DEV), gain.to(DEV)
    out, stats = torch.empty(1, t, d, device=DEV, dtype=dtype), torch.empty(2, n, t, device=DEV)
    _lib.check(_lib.lib().sy_fwd_gain(vd.data_ptr(), wd.data_ptr(), gd.data_ptr(), out.data_ptr(), stats.data_ptr(),
                                      n, t, d, t * d, _lib.dtype_code(dtype), _lib.dtype_code(dtype), 1e-6,
                                      _lib.stream_ptr(vd.device)), "sy_fwd_gain")
    r = torch.rsqrt(v.double().square().mean(-1) + 1e-6)[:, 0]
    assert rel_l2(stats[0], (v.double() @ (w.double() * gain.double()))[:, 0] * r) <= 2e-6 and out.isfinite().all()
