"""Queries of another dtype than the sources (a module's fp32 parameters with
16-bit activations, and the other mixes) on the vector kernels: forward, the
statistics variant and every backward family at the tiles' edges, against the
float64 oracle at the bars of a query of the sources' dtype."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle import c_oracle  # noqa: E402
from oracle.reference import block_attn_res_oracle, dtype_floor, oracle_grads, rel_l2  # noqa: E402
from switchyard import _lib  # noqa: E402
from switchyard.stats_op import attn_with_stats  # noqa: E402
from switchyard.table_op import block_attn_res_sources  # noqa: E402
from switchyard.triton_op import block_attn_res_triton  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32

# (N, T, D): one- to eight-wave rows, partial chunks of the last lane, each row
# tile's last and first count, chunked forwards, the tall backward tiles, few
# tokens per CU (the token rule's tiles) and several tokens a slot.
SHAPES = [(9, 1100, 2048), (1, 5, 64), (4, 33, 1024), (5, 40, 4096), (9, 24, 8192), (16, 70, 2048),
          (10, 1600, 2048), (17, 48, 2048), (32, 40, 1024), (33, 24, 1024), (7, 33, 328), (3, 8, 16384),
          (9, 600, 1544)]


def _bar(ref, dtype):
    # 16-bit: one rounding of each output. fp32: the bar of the fp32 gradients.
    return 1e-5 if dtype == F else 1.10 * dtype_floor(ref, dtype)


def _inputs(n, t, d, vdt, wdt, seed=0):
    g = torch.Generator().manual_seed(seed)
    v = torch.randn(n, 1, t, d, generator=g).to(vdt)
    w = (torch.randn(d, generator=g) * d**-0.5).to(wdt)
    go = torch.randn(1, t, d, generator=g).to(vdt)
    return v, w, go


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtypes", [(BF, F), (HF, F), (BF, HF), (F, BF)])
def test_query_of_another_dtype(shape, dtypes):
    vdt, wdt = dtypes
    n, t, d = shape
    print(f"mixed {shape} {vdt} {wdt}", flush=True)
    v, w, go = _inputs(n, t, d, vdt, wdt)
    vv, ww = v.to(DEV).requires_grad_(), w.to(DEV).requires_grad_()
    out = block_attn_res_triton(vv, ww)
    dv, dw = torch.autograd.grad(out, (vv, ww), go.to(DEV))
    assert out.dtype == dv.dtype == vdt and dw.dtype == wdt
    ro = block_attn_res_oracle(v, w)
    rdv, rdw = oracle_grads(v, w, go)
    assert rel_l2(out.detach(), ro) <= _bar(ro, vdt)
    assert rel_l2(dv, rdv) <= _bar(rdv, vdt)
    if n > 1:  # one source: alpha is 1 and dw is zero
        assert rel_l2(dw, rdw) <= _bar(rdw, wdt)
    else:
        assert torch.count_nonzero(dw) == 0


@pytest.mark.parametrize("dtypes", [(BF, F), (F, HF)])
def test_mixed_sources_and_statistics(dtypes):
    """The pointer-list and (o, m, l) variants of the same tiles."""
    vdt, wdt = dtypes
    n, t, d = 9, 300, 2048
    v, w, go = _inputs(n, t, d, vdt, wdt, seed=3)
    ww = w.to(DEV).requires_grad_()
    vs = [x.to(DEV).requires_grad_() for x in v]
    stacked = v.to(DEV).requires_grad_()
    grads = torch.autograd.grad(block_attn_res_sources(vs, ww), [*vs, ww], go.to(DEV))
    ref = torch.autograd.grad(block_attn_res_triton(stacked, ww), (stacked, ww), go.to(DEV))
    assert all(torch.equal(a, b) for a, b in zip(grads[:n], ref[0])) and torch.equal(grads[n], ref[1])

    g = torch.Generator().manual_seed(5)
    gm, gl = torch.randn(1, t, generator=g), torch.randn(1, t, generator=g)
    o, m, ell = attn_with_stats(stacked, ww)
    dv, dw = torch.autograd.grad((o, m, ell), (stacked, ww), (go.to(DEV), gm.to(DEV), gl.to(DEV)))
    np64 = [x.double().numpy() for x in (v[:, 0], w, go[0], gm[0], gl[0])]
    ro, rm, rl = (torch.from_numpy(x) for x in c_oracle.attn_with_stats(*np64[:2]))
    rdv, rdw = (torch.from_numpy(x) for x in c_oracle.attn_with_stats_backward(*np64))
    assert rel_l2(o[0].detach().cpu(), ro) <= _bar(ro, vdt)
    assert rel_l2(m[0].detach().cpu(), rm) <= 1e-5 and rel_l2(ell[0].detach().cpu(), rl) <= 1e-5
    assert rel_l2(dv[:, 0].cpu(), rdv) <= _bar(rdv, vdt)
    assert rel_l2(dw.cpu(), rdw) <= _bar(rdw, wdt)


def test_the_launched_plan_of_a_mixed_query():
    """An fp32 query runs the sources' tiles; a 16-bit row of more than 1024
    chunks keeps the element-wise backward (its tile holds the query packed)."""
    assert _lib.plan(_lib.OP_FWD, 9, 2048, BF, w_dtype=F, n_tok=4096)["family_name"] == "resident"
    assert _lib.plan(_lib.OP_BWD, 9, 2048, BF, w_dtype=F, n_tok=4096)["family_name"] == "resident"
    assert _lib.plan(_lib.OP_BWD, 9, 16384, BF, w_dtype=F, n_tok=64)["family_name"] == "generic"
    assert _lib.plan(_lib.OP_FWD, 9, 7, BF, w_dtype=F, n_tok=64)["family_name"] == "generic"
