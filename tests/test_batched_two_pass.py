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
