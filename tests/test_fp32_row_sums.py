"""fp32 gradients against float64 where a row's sums are formed by matrix products or by one
lane over several chunks: the error stays that of short chains.

Bound: a chain of k additions errs by about sqrt(k) * 2^-24 / 2 of its terms' norm, and the
logits pass it on to the gradients times their own size, here queries of 0.5 N(0, 1): twice
that scale doubles every figure. So scaled, short chains and a tree measured 1.1e-6, 0.5e-6
and 0.6e-6 on the cases below; one running sum over a lane's share 2.2e-6 on the first."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle.reference import rel_l2  # noqa: E402
from switchyard.hip_op import block_attn_res_batched_train, block_attn_res_hip  # noqa: E402


def _f64(v, q):
    r = torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-6)
    out = []
    for row in q:
        p = torch.softmax((v * r * row).sum(-1), 0)
        out.append((p.unsqueeze(-1) * v).sum(0))
    return torch.stack(out)


# (N, S, T, D, bound); S = 0: the operator itself, on rows no 16-byte load can start at
CASES = [(11, 4, 1262, 1024, 1.6e-6), (9, 8, 2048, 256, 0.8e-6), (5, 0, 1500, 777, 0.8e-6)]


@pytest.mark.parametrize("case", CASES)
def test_fp32_gradient_error(case):
    n, s, t, d, bound = case
    print(f"fp32 sums {case}", flush=True)
    g = torch.Generator().manual_seed(n + d)
    v = torch.randn(n, 1, t, d, generator=g)
    q = 0.5 * torch.randn(max(s, 1), d, generator=g)
    go = torch.randn(max(s, 1), 1, t, d, generator=g)
    vd, qd = v.double().requires_grad_(), q.double().requires_grad_()
    ref = torch.autograd.grad(_f64(vd, qd), (vd, qd), go.double())
    vg, qg = v.cuda().requires_grad_(), q.cuda().requires_grad_()
    out = block_attn_res_batched_train(vg, qg) if s else block_attn_res_hip(vg, qg[0]).unsqueeze(0)
    got = torch.autograd.grad(out, (vg, qg), go.cuda())
    errs = [float(rel_l2(a.cpu(), b)) for a, b in zip(got, ref)]
    print(errs, flush=True)
    assert max(errs) <= bound, errs
