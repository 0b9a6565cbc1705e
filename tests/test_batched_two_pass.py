"""The two-pass batched backward (rows of whole 16-byte chunks, up to 16 sources and
16 queries, where the matrix-core single pass does not apply) against the C oracle:
every row and query group's first and last count, a row of one chunk, partial chunks
and partial steps, one token, and several tokens a group."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle import c_oracle  # noqa: E402
from oracle.reference import dtype_floor, rel_l2  # noqa: E402
from switchyard import _lib  # noqa: E402
from switchyard.hip_op import block_attn_res_batched_train  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32

# (N, S, T, D)
CASES = [(9, 8, 300, 4096), (4, 4, 37, 4096), (5, 5, 1, 2056), (10, 9, 40, 2048), (16, 16, 33, 1032),
         (1, 8, 12, 320), (2, 1, 700, 64), (9, 3, 65, 8), (16, 8, 20, 2048), (3, 12, 3000, 128),
         (12, 4, 50, 6144)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [BF, HF, F])
def test_two_pass_batched_backward(case, dtype):
    n, s, t, d = case
    print(f"two-pass batched bwd {case} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(n * s + d)
    v = torch.randn(n, 1, t, d, generator=gen).to(dtype)
    q = (torch.randn(s, d, generator=gen) * 2.0 / d**0.5).to(dtype)
    g = torch.randn(s, 1, t, d, generator=gen).to(dtype)
    vv, qq = v.to(DEV).requires_grad_(), q.to(DEV).requires_grad_()
    runs = [torch.autograd.grad(block_attn_res_batched_train(vv, qq), (vv, qq), g.to(DEV)) for _ in range(2)]
    assert all(torch.equal(a, b) for a, b in zip(*runs))  # fixed-order sums
    np64 = [x.double().numpy() for x in (v[:, 0], q, g[:, 0])]
    rdv, rdq = (torch.from_numpy(x) for x in c_oracle.batched_backward(*np64))
    dv, dq = (x.cpu() for x in runs[0])
    bar = (lambda ref: 1e-5) if dtype == F else (lambda ref: 1.10 * dtype_floor(ref, dtype))
    assert rel_l2(dv[:, 0], rdv) <= bar(rdv)
    if n == 1:  # one source: its weight is 1 whatever the query
        assert not dq.any()
    else:
        assert rel_l2(dq, rdq) <= bar(rdq)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [BF, HF, F])
def test_what_is_launched(case, dtype):
    n, s, t, d = case
    few = {(1, 8, 12, 320), (2, 1, 700, 64), (9, 3, 65, 8)}  # few queries keep the register tile,
    small = {(4, 4, 37, 4096), (5, 5, 1, 2056)}  # 16-bit ones also at few tokens
    family = _lib.plan(_lib.OP_BWD_BATCHED, n, d, dtype, n_q=s, n_tok=t)["family_name"]
    assert (family == "two_pass") == (case not in few and not (dtype != F and case in small))


def test_a_workspace_too_small_for_two_passes():
    """A source stride past the matrix kernel's offsets, with the workspace sized for that
    kernel, runs the register tile (at this many tokens the coefficients do not fit); with
    room for them two passes; with room for neither it is refused. Nothing is written past
    the workspace."""
    n, s, t, d = 9, 8, 7000, 512
    stride = 400 << 20  # elements; the matrix kernel adds three to a 31-bit byte offset
    gen = torch.Generator().manual_seed(1)
    v, q = torch.randn(n, t, d, generator=gen).to(BF), (torch.randn(s, d, generator=gen) * 2.0 / d**0.5).to(BF)
    g = torch.randn(s, t, d, generator=gen).to(BF)
    buf = torch.empty((n - 1) * stride + t * d, device=DEV, dtype=BF)
    for k in range(n):
        buf[k * stride : k * stride + t * d].copy_(v[k].flatten())
    qd, gd = q.to(DEV), g.to(DEV)
    need = _lib.lib().sy_bwd_batched_workspace_bytes(n, s, t, d, _lib.dtype_code(BF))
    rdv, rdq = (torch.from_numpy(x) for x in c_oracle.batched_backward(*[x.double().numpy() for x in (v, q, g)]))
    got = []
    for size in (64 << 20, need, s * d * 4 - 16):
        print(f"two-pass workspace {size}", flush=True)
        dv, dq = torch.empty(n, t, d, device=DEV, dtype=BF), torch.empty(s, d, device=DEV, dtype=BF)
        ws = torch.full((size // 4 + 1024,), 7.0, device=DEV)
        rc = _lib.lib().sy_bwd_batched(buf.data_ptr(), qd.data_ptr(), gd.data_ptr(), dv.data_ptr(), dq.data_ptr(),
                                       ws.data_ptr(), size, n, s, t, d, stride, _lib.dtype_code(BF), 1e-6,
                                       _lib.stream_ptr(buf.device))
        assert (ws[size // 4 :] == 7.0).all()
        if size < need:
            assert rc < 0
            continue
        assert rc == 0
        assert rel_l2(dv.cpu(), rdv) <= 1.10 * dtype_floor(rdv, BF) and rel_l2(dq.cpu(), rdq) <= 1.10 * dtype_floor(rdq, BF)
        got.append(dv)
    assert not torch.equal(*got)  # two kernels, two orders of sums
