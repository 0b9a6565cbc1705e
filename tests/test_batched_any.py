"""The batched forward for any row (k_batched_any: shapes the matrix-core and register
kernels do not take) with its statistics, against the C oracle: every row and query
group's first and last count, one chunk, partial chunks and steps, misaligned buffers."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

from oracle import c_oracle  # noqa: E402
from oracle.reference import dtype_floor, rel_l2  # noqa: E402
from switchyard import _lib  # noqa: E402
from switchyard.hip_op import block_attn_res_batched  # noqa: E402
from switchyard.stats_op import block_attn_res_batched_with_stats  # noqa: E402

DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32

# (N, S, T, D)
CASES = [(12, 8, 300, 1280), (9, 8, 1500, 256), (9, 8, 70, 2560), (10, 9, 40, 2056), (16, 16, 33, 1032), (4, 4, 37, 777),
         (5, 5, 1, 2313), (1, 8, 12, 320), (9, 16, 65, 8), (3, 12, 3000, 129), (12, 4, 50, 6151), (9, 10, 9, 4097),
         (16, 1, 21, 63), (12, 3, 20, 8192)]


def _inputs(n, s, t, d, dtype):
    g = torch.Generator().manual_seed(n * s + d)
    v = torch.randn(n, 1, t, d, generator=g).to(dtype)
    return v, (torch.randn(s, d, generator=g) * 2.0 / d**0.5).to(dtype)


def _bar(ref, dtype):
    return 1e-5 if dtype == F else 1.10 * dtype_floor(ref, dtype)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [BF, HF, F])
def test_batched_forward_and_statistics(case, dtype):
    n, s, t, d = case
    print(f"batched any {case} {dtype}", flush=True)
    v, q = _inputs(*case, dtype)
    ref = torch.from_numpy(c_oracle.batched(v[:, 0].double().numpy(), q.double().numpy()))
    out = block_attn_res_batched(v.to(DEV), q.to(DEV))
    assert rel_l2(out[:, 0].cpu(), ref) <= _bar(ref, dtype)
    o, m, ell = block_attn_res_batched_with_stats(v.to(DEV), q.to(DEV))
    for k in range(s):
        ro, rm, rl = (torch.from_numpy(x) for x in c_oracle.attn_with_stats(v[:, 0].double().numpy(), q[k].double().numpy()))
        assert rel_l2(o[k, 0].cpu(), ro) <= _bar(ro, dtype)
        assert rel_l2(m[k, 0].cpu(), rm) <= 1e-5 and rel_l2(ell[k, 0].cpu(), rl) <= 1e-5


@pytest.mark.parametrize("dtype", [BF, F])
def test_misaligned_buffers_and_guards(dtype):
    import ctypes

    from switchyard import _lib

    n, s, t, d = 9, 8, 33, 1280
    v, q = _inputs(n, s, t, d, dtype)

    def off(x):
        buf = torch.empty(x.numel() + 1, device=DEV, dtype=x.dtype)
        return buf[1:].view_as(x).copy_(x)

    vm, qm = off(v), off(q)
    buf = torch.full((s * t * d + 64,), 7.0, device=DEV, dtype=dtype)
    out, P = buf[31:], lambda x: ctypes.c_void_p(x.data_ptr())
    rc = _lib.lib().sy_fwd_batched(P(vm), P(qm), P(out), n, s, t, d, t * d, _lib.dtype_code(dtype), 1e-6,
                                   _lib.stream_ptr(vm.device))
    assert rc == 0
    torch.cuda.synchronize()
    ref = torch.from_numpy(c_oracle.batched(v[:, 0].double().numpy(), q.double().numpy()))
    assert rel_l2(out[: s * t * d].view(s, t, d).cpu(), ref) <= _bar(ref, dtype)
    assert bool((buf[:31] == 7).all()) and bool((buf[31 + s * t * d:] == 7).all())


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [BF, HF, F])
def test_what_is_launched(case, dtype):
    n, s, t, d = case
    few = {(1, 8, 12, 320), (16, 1, 21, 63)}  # too few pairs, too few queries
    tiles = {(9, 8, 1500, 256), (9, 8, 70, 2560), (9, 16, 65, 8)}  # fp32 of up to nine rows
    family = _lib.plan(_lib.OP_BATCHED, n, d, dtype, n_q=s, n_tok=t)["family_name"]
    assert (family == "stream") == (case not in few and not (dtype == F and case in tiles))
