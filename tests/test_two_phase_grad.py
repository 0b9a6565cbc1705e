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
