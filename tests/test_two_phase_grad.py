"""The two-phase schedule's gradient in one pass over the sources: both phases
fill one statistics array, at every split that changes a phase's tile or sends
phase 2 to the unfused merge, against the float64 oracle."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle.reference import block_attn_res_oracle, dtype_floor, oracle_grads, rel_l2  # noqa: E402
from switchyard import stats_op  # noqa: E402
from switchyard.stats_op import block_attn_res_two_phase  # noqa: E402

DEV = "cuda"
BF, F = torch.bfloat16, torch.float32

# (N, split, T, D): one-row phases, the last resident merge tile (15 sources and
# the prior), the unfused merge (16 and more, odd rows), chunked phase 1.
CASES = [(2, 1, 5, 64), (9, 4, 1100, 2048), (9, 8, 70, 2048), (16, 1, 40, 1024), (17, 1, 40, 1024),
         (20, 17, 33, 1024), (12, 3, 24, 4096), (5, 2, 33, 777)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtypes", [(BF, BF), (F, F), (BF, F)])
def test_two_phase_output_and_gradients(case, dtypes):
    vdt, wdt = dtypes
    n, split, t, d = case
    print(f"two phase {case} {vdt} {wdt}", flush=True)
    g = torch.Generator().manual_seed(n + d)
    v = torch.randn(n, 1, t, d, generator=g).to(vdt)
    w = (torch.randn(d, generator=g) * d**-0.5).to(wdt)
    go = torch.randn(1, t, d, generator=g).to(vdt)
    vv, ww = v.to(DEV).requires_grad_(), w.to(DEV).requires_grad_()
    out = block_attn_res_two_phase(vv, ww, split)
    dv, dw = torch.autograd.grad(out, (vv, ww), go.to(DEV))
    ro = block_attn_res_oracle(v, w)
    # The partial result is rounded before the merge: three roundings.
    assert rel_l2(out.detach(), ro) <= (1e-5 if vdt == F else 2.5 * dtype_floor(ro, vdt))
    for got, ref, dt in zip((dv, dw), oracle_grads(v, w, go), (vdt, wdt)):
        assert rel_l2(got, ref) <= (1e-5 if dt == F else 1.10 * dtype_floor(ref, dt))


# Where the union's backward is element-wise and the groups' are not, and its neighbours:
# (N, split, T, D, by groups).
ROUTES = [(17, 8, 9000, 64, True), (17, 8, 8192, 64, False), (24, 12, 9000, 512, True), (20, 3, 9000, 128, False),
          (20, 10, 512, 4160, True), (20, 10, 40, 8192, True), (20, 10, 40, 4160, False), (16, 8, 600, 4104, False),
          (10, 5, 520, 8200, True), (33, 16, 9000, 128, False)]


@pytest.mark.parametrize("case", ROUTES)
def test_routes_of_the_gradient(case):
    n, split, t, d, groups = case
    print(f"two phase route {case}", flush=True)
    g = torch.Generator().manual_seed(n + d)
    v, go = torch.randn(n, 1, t, d, generator=g).to(BF), torch.randn(1, t, d, generator=g).to(BF)
    w = (torch.randn(d, generator=g) * d**-0.5).to(BF)
    vv, ww = v.to(DEV).requires_grad_(), w.to(DEV).requires_grad_()
    assert stats_op._by_groups(vv, ww, split) == groups
    assert not stats_op._by_groups(vv.detach(), ww.detach(), split)
    out = block_attn_res_two_phase(vv, ww, split)
    assert ("TwoPhase" in out.grad_fn.name()) != groups
    dv, dw = torch.autograd.grad(out, (vv, ww), go.to(DEV))
    with torch.no_grad():
        assert torch.equal(block_attn_res_two_phase(vv, ww, split), out)
    ro = block_attn_res_oracle(v, w)
    assert rel_l2(out.detach(), ro) <= 2.5 * dtype_floor(ro, BF)
    # by groups the partial results' gradients are rounded too: four roundings
    for got, ref in zip((dv, dw), oracle_grads(v, w, go)):
        assert rel_l2(got, ref) <= (3.5 if groups else 1.10) * dtype_floor(ref, BF)


def test_more_sources_than_one_launch_takes():
    """4096 is the most of one element-wise launch: the two groups' gradients, in fp32."""
    g = torch.Generator().manual_seed(0)
    v, go, w = torch.randn(4100, 1, 2, 8, generator=g), torch.randn(1, 2, 8, generator=g), torch.randn(8, generator=g)
    vv, ww = v.to(DEV).requires_grad_(), w.to(DEV).requires_grad_()
    out = block_attn_res_two_phase(vv, ww, 2050)
    for got, ref in zip(torch.autograd.grad(out, (vv, ww), go.to(DEV)), oracle_grads(v, w, go)):
        assert rel_l2(got, ref) <= 1e-4  # sums of 4100 terms, through partial results of 2050
