"""Rows that are not whole 16-byte chunks at 16-byte boundaries (odd widths, buffers
one element off) on the unaligned kernels: every tile's first and last width, a row of
one chunk and one element more, row counts at the tiles' edges, and neighbours that a
store past a row's end would damage; against the float64 oracle."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle.reference import block_attn_res_oracle, dtype_floor, oracle_grads, rel_l2  # noqa: E402
from switchyard import _lib  # noqa: E402
from switchyard.table_op import block_attn_res_sources  # noqa: E402
from switchyard.triton_op import block_attn_res_triton  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32

# (N, T, D): 16-bit chunk counts 2, 64/65 (one slot / two), 128/129, 256/257, 512/513,
# 1024; fp32 has twice as many. D = 7 and 8193 (16-bit) stay element-wise.
SHAPES = [(5, 1023, 777), (9, 1100, 63), (4, 37, 9), (10, 33, 511), (16, 40, 513), (9, 29, 1023), (3, 50, 1025),
          (9, 21, 2047), (17, 25, 2049), (33, 9, 777), (2, 11, 4095), (5, 9, 4097), (9, 5, 8191), (4, 20, 7),
          (2, 3, 8193), (12, 1, 129)]


def _bar(ref, dtype):
    return 1e-5 if dtype == F else 1.10 * dtype_floor(ref, dtype)


def _inputs(n, t, d, vdt, wdt, seed=0):
    g = torch.Generator().manual_seed(seed)
    v = torch.randn(n, 1, t, d, generator=g).to(vdt)
    w = (torch.randn(d, generator=g) * d**-0.5).to(wdt)
    return v, w, torch.randn(1, t, d, generator=g).to(vdt)


def _check(out, dv, dw, v, w, go):
    for got, ref, dt in ((out, block_attn_res_oracle(v, w), v.dtype), *zip((dv, dw), oracle_grads(v, w, go), (v.dtype, w.dtype))):
        assert rel_l2(got.detach(), ref) <= _bar(ref, dt)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtypes", [(BF, BF), (HF, HF), (F, F), (BF, F)])
def test_odd_widths(shape, dtypes):
    print(f"unaligned {shape} {dtypes}", flush=True)
    v, w, go = _inputs(*shape, *dtypes)
    vv, ww = v.to(DEV).requires_grad_(), w.to(DEV).requires_grad_()
    out = block_attn_res_triton(vv, ww)
    _check(out, *torch.autograd.grad(out, (vv, ww), go.to(DEV)), v, w, go)


@pytest.mark.parametrize("shape", [(9, 70, 2048), (4, 33, 512), (16, 20, 1024), (5, 19, 777)])
@pytest.mark.parametrize("dtype", [BF, F])
def test_misaligned_buffers(shape, dtype):
    """Sources, query and gradient each one element past a 16-byte boundary."""
    n, t, d = shape
    v, w, go = _inputs(n, t, d, dtype, dtype, seed=2)

    def off(x):
        buf = torch.empty(x.numel() + 1, device=DEV, dtype=x.dtype)
        return buf[1:].view_as(x).copy_(x)

    vs = [off(x).requires_grad_() for x in v]
    ww, gg = off(w).requires_grad_(), off(go)
    out = block_attn_res_sources(vs, ww)
    *dvs, dw = torch.autograd.grad(out, [*vs, ww], gg)
    _check(out, torch.stack(dvs), dw, v, w, go)
    stacked = off(v).requires_grad_()
    out = block_attn_res_triton(stacked, ww)
    dv, dw = torch.autograd.grad(out, (stacked, ww), gg)
    _check(out, dv, dw, v, w, go)


def test_stores_stay_inside_the_rows():
    """Output and gradient rows between guard elements keep the guards."""
    import ctypes

    n, t, d = 5, 31, 777
    v, w, go = (x.to(DEV) for x in _inputs(n, t, d, HF, HF, seed=4))
    lib, P = _lib.lib(), lambda x: ctypes.c_void_p(x.data_ptr())
    out = torch.full((t * d + 64,), 7.0, device=DEV, dtype=HF)
    dv = torch.full((n * t * d + 64,), 7.0, device=DEV, dtype=HF)
    stats = torch.empty(2, n, t, device=DEV)
    dw = torch.empty(d, device=DEV, dtype=HF)
    bytes_ = lib.sy_bwd_workspace_bytes(n, t, d, 1, 1)
    ws = torch.full((bytes_ // 4 + 64,), 7.0, device=DEV)
    st = _lib.stream_ptr(v.device)
    o, g = out[31:], dv[31:]  # odd starts, 31 and 33 guards
    assert lib.sy_fwd(P(v), P(w), P(o), P(stats), n, t, d, t * d, 1, 1, 1e-6, st) == 0
    assert lib.sy_bwd(P(v), P(w), P(go), P(stats), P(g), P(dw), P(ws), bytes_, n, t, d, t * d, 1, 1, 1e-6, st) == 0
    torch.cuda.synchronize()
    for buf, size in ((out, t * d), (dv, n * t * d)):
        assert bool((buf[:31] == 7).all()) and bool((buf[31 + size:] == 7).all())
    assert bool((ws[bytes_ // 4:] == 7).all())
    _check(o[: t * d].view(1, t, d), g[: n * t * d].view(n, 1, t, d), dw, v.cpu(), w.cpu(), go.cpu())


def test_the_launched_plan_of_unaligned_rows():
    p = _lib.plan(_lib.OP_FWD, 5, 777, HF, n_tok=1023)
    assert (p["waves_per_token"], p["chunks_per_lane"], p["rows_per_tile"]) == (1, 2, 9)
    p = _lib.plan(_lib.OP_BWD, 16, 8191, HF, n_tok=64)
    assert (p["waves_per_token"], p["chunks_per_lane"], p["rows_per_tile"]) == (8, 2, 16)
    for n, d in ((5, 7), (5, 8193)):
        assert _lib.plan(_lib.OP_FWD, n, d, HF, n_tok=64)["family_name"] == "generic"
    assert _lib.plan(_lib.OP_BWD, 17, 777, HF, n_tok=64)["family_name"] == "generic"
