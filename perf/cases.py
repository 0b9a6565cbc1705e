"""The work this framework is measured on: each case is one call, or one
forward + backward, through a public entry point of ``switchyard``.

``listed()`` holds the cases, ``draw(rng)`` more of the same ranges. For one case,
``prepare`` makes what a caller holds before the call, ``run`` makes the call,
``work`` counts the bytes and operations it cannot do without, ``exact`` gives the
same outputs in float64 without this framework's code, and ``tolerance`` says how
far another correct implementation at the same precision may be off.
"""

from __future__ import annotations

import math
import pathlib
import sys

import torch

_PKG = pathlib.Path(__file__).resolve().parent.parent / "blackwell-switchyard_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

EPS = 1e-6
DEV = "cuda"
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # One decoded token of eight sequences: latency and launches are all there is.
        dict(name="decode", kind="op", grad=False, n=9, b=8, t=1, d=2048, dtype="bf16"),
        # The fp32 plumbing configuration, forward and backward.
        dict(name="small_fp32", kind="op", grad=True, n=4, b=1, t=256, d=512, dtype="fp32"),
        # The operator's representative training shape.
        dict(name="representative", kind="op", grad=True, n=9, b=1, t=4096, d=2048, dtype="bf16"),
        # A deep model's late sites: 32 sources.
        dict(name="deep", kind="op", grad=True, n=32, b=1, t=4096, d=2048, dtype="bf16"),
        # The widest batch of the D sweep.
        dict(name="wide", kind="op", grad=True, n=9, b=4, t=4096, d=4096, dtype="bf16"),
        # Mixed-precision training: the module keeps its parameters in fp32, the
        # activations are bf16.
        dict(name="module_mixed", kind="module", grad=True, n=9, b=2, t=2048, d=2048, dtype="bf16"),
        # Ragged everything: a row that is no multiple of 16 bytes, odd B and T.
        dict(name="ragged", kind="op", grad=True, n=5, b=3, t=341, d=777, dtype="fp16"),
        # A site of the 1.3B decoder's training step (batch 4 x 2048) whose sources
        # are separate tensors.
        dict(name="sources", kind="sources", grad=True, n=8, b=4, t=2048, d=2048, dtype="bf16"),
        # Eight queries against one read of the sources, output only.
        dict(name="batched", kind="batched", grad=False, n=9, s=8, b=1, t=4096, d=2048, dtype="bf16"),
        # The same trained, at twice the width.
        dict(name="batched_train", kind="batched", grad=True, n=9, s=8, b=1, t=4096, d=4096, dtype="bf16"),
        # The two-phase schedule trained: four inter-block and five intra-block sources.
        dict(name="two_phase", kind="two_phase", grad=True, n=9, split=4, b=1, t=4096, d=2048, dtype="bf16"),
        # Prefill of the small decoder: a whole call, logits out.
        dict(name="model_prefill", kind="model", grad=False, layers=8, blocks=4, heads=8, vocab=4096,
             d_ff=1408, b=4, t=512, d=512, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _slab_bytes(c):
    return c["b"] * c["t"] * c["d"] * _SIZE[c["dtype"]]


def draw(rng):
    kind = rng.choice(["op", "op", "op", "op", "module", "module", "sources", "batched", "batched", "two_phase", "model"])
    if kind == "model":
        d = 64 * rng.randint(4, 12)
        return dict(kind=kind, grad=False, layers=2 * rng.randint(1, 4), blocks=rng.choice([2, 4]), heads=d // 64,
                    vocab=rng.choice([1000, 4096]), d_ff=64 * rng.randint(8, 24), b=rng.randint(1, 4),
                    t=_log(rng, 32, 512), d=d, dtype="bf16")
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    if kind == "module":
        dtype = rng.choice(["bf16", "bf16", "fp16"])
    # Widths: mostly multiples of 64, some of them powers of two, one in six odd.
    how = rng.random()
    d = 2 ** rng.randint(8, 13) if how < 0.4 else 64 * _log(rng, 4, 96)
    if how > 0.83:
        d = _log(rng, 65, 4000) | 1
    top = {"op": 33, "module": 16, "sources": 16, "batched": 12, "two_phase": 16}[kind]
    c = dict(kind=kind, grad=rng.random() < 0.7, n=_log(rng, 2, top),
             b=rng.choice([1, 1, 2, 3, 4, 8]), t=_log(rng, 1, 8192), d=d, dtype=dtype)
    slabs = 3 * c["n"] + 2
    if kind == "batched":
        c["s"] = rng.randint(1, 10)
        slabs = 3 * c["n"] + 3 * c["s"]
    if kind == "two_phase":
        c["split"] = rng.randint(1, c["n"] - 1)
    # Element-wise rows are an order of magnitude slower: keep them smaller.
    most = 2.0e9 if d % 8 == 0 else 2.0e8
    while c["t"] > 1 and slabs * _slab_bytes(c) > most:
        c["t"] = max(1, c["t"] // 2)
    return c


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _inputs(c, seed):
    """Sources v ~ N(0,1), queries ~ N(0, 0.5), output gradients ~ N(0,1)."""
    g, dt = _gen(seed), _DT[c["dtype"]]
    n, b, t, d = c["n"], c["b"], c["t"], c["d"]
    x = {"v": torch.randn(n, b, t, d, device=DEV, dtype=dt, generator=g)}
    if c["kind"] == "module":
        x["w"] = 0.5 * torch.randn(d, device=DEV, generator=g)
        x["gain"] = 1.0 + 0.1 * torch.randn(d, device=DEV, generator=g)
    elif c["kind"] == "batched":
        x["w"] = (0.5 * torch.randn(c["s"], d, device=DEV, generator=g)).to(dt)
    else:
        x["w"] = (0.5 * torch.randn(d, device=DEV, generator=g)).to(dt)
    if c["grad"]:
        shape = (c["s"], b, t, d) if c["kind"] == "batched" else (b, t, d)
        x["g"] = torch.randn(shape, device=DEV, dtype=dt, generator=g)
    return x


def _model_inputs(c, seed):
    """Weights of a decoder as trained ones are scaled, and token ids."""
    g, d, ff = _gen(seed), c["d"], c["d_ff"]

    def normal(std, *shape):
        return (std * torch.randn(*shape, device=DEV, generator=g)).to(torch.bfloat16)

    w = {"embed.weight": normal(1.0, c["vocab"], d)}
    for i in range(c["layers"]):
        p = f"layers.{i}."
        w[p + "attn_norm.weight"] = 1 + normal(0.1, d)
        w[p + "attn.qkv.weight"] = normal(d**-0.5, 3 * d, d)
        w[p + "attn.out.weight"] = normal(d**-0.5, d, d)
        w[p + "mlp_norm.weight"] = 1 + normal(0.1, d)
        w[p + "mlp.gate_up.weight"] = normal(d**-0.5, 2 * ff, d)
        w[p + "mlp.down.weight"] = normal(ff**-0.5, d, ff)
    for i in range(2 * c["layers"] + 1):
        w[f"attn_res.{i}.w"] = normal(0.5 * d**-0.5, d)
        w[f"attn_res.{i}.g"] = 1 + normal(0.1, d)
    w["final_norm.weight"] = 1 + normal(0.1, d)
    w["lm_head.weight"] = normal(d**-0.5, c["vocab"], d)
    return w, torch.randint(0, c["vocab"], (c["b"], c["t"]), device=DEV, generator=g)


def prepare(case, seed):
    c = case
    if c["kind"] == "model":
        from switchyard.model import ModelConfig, Transformer

        w, idx = _model_inputs(c, seed)
        cfg = ModelConfig(vocab_size=c["vocab"], d_model=c["d"], n_layers=c["layers"], n_heads=c["heads"],
                          d_ff=c["d_ff"], n_blocks=c["blocks"], max_seq_len=512, tie_embeddings=False,
                          residual="switchyard")
        with torch.device(DEV):
            model = Transformer(cfg)
        model.load_state_dict(w)
        # The rotary tables stay fp32, as the model's own precision policy has it.
        for p in model.parameters():
            p.data = p.data.to(torch.bfloat16)
        return {"case": c, "model": model, "idx": idx}
    x = _inputs(c, seed)
    s = {"case": c, "g": x.get("g")}
    if c["kind"] == "module":
        from switchyard.triton_op import BlockAttnResTriton

        mod = BlockAttnResTriton(c["d"]).to(DEV)
        with torch.no_grad():
            mod.w.copy_(x["w"])
            mod.g.copy_(x["gain"])
        s["mod"] = mod
    else:
        s["w"] = x["w"].requires_grad_(c["grad"])
    if c["kind"] == "sources":
        s["v"] = [v.clone().requires_grad_(c["grad"]) for v in x["v"]]
    else:
        s["v"] = x["v"].requires_grad_(c["grad"])
    return s


# --------------------------------------------------------------- the calls


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "model":
        with torch.no_grad():
            return {"logits": state["model"](state["idx"])}
    with torch.set_grad_enabled(c["grad"]):
        if kind == "op":
            from switchyard.triton_op import block_attn_res_triton

            leaves = [state["v"], state["w"]]
            out = block_attn_res_triton(state["v"], state["w"], EPS)
        elif kind == "module":
            leaves = [state["v"], state["mod"].w, state["mod"].g]
            out = state["mod"](state["v"])
        elif kind == "sources":
            from switchyard.table_op import block_attn_res_sources

            leaves = [*state["v"], state["w"]]
            out = block_attn_res_sources(state["v"], state["w"], EPS)
        elif kind == "batched":
            from switchyard.hip_op import block_attn_res_batched_train
            from switchyard.triton_op import block_attn_res_batched

            leaves = [state["v"], state["w"]]
            op = block_attn_res_batched_train if c["grad"] else block_attn_res_batched
            out = op(state["v"], state["w"], EPS)
        else:
            from switchyard.stats_op import block_attn_res_two_phase

            leaves = [state["v"], state["w"]]
            out = block_attn_res_two_phase(state["v"], state["w"], c["split"], EPS)
    if not c["grad"]:
        return {"out": out}
    return {"out": out.detach(), "grads": list(torch.autograd.grad(out, leaves, state["g"]))}


# -------------------------------------------------------- what is expected


def work(case):
    c = case
    if c["kind"] == "model":
        d, tok, nl = c["d"], c["b"] * c["t"], c["layers"]
        params = nl * (4 * d * d + 3 * d * c["d_ff"]) + c["vocab"] * d
        flops = 2 * tok * params + nl * 2 * tok * c["t"] * d
        # Every sublayer reads the weights once and moves its activations and the
        # residual site's sources; the logits are written once.
        size = c["blocks"]
        per = 2 * nl // size
        sources = sum((j + 1) + (j + 2) * (per - 1) for j in range(size)) + size + 1
        return {"bytes": 2 * (params + tok * d * (sources + 2 * nl * 4) + tok * c["vocab"]), "flops": flops}
    n, s = c["n"], c.get("s", 1)
    slab = _slab_bytes(c)
    elems = c["b"] * c["t"] * c["d"]
    # Forward: read the sources, write the outputs. Backward: read the sources and
    # the output gradients, write the source gradients.
    slabs = n + s + (2 * n + s if c["grad"] else 0)
    flops = elems * n * s * (6 + (10 if c["grad"] else 0))
    return {"bytes": slabs * slab + 2 * s * c["d"] * _SIZE[c["dtype"]], "flops": flops}


def tolerance(case):
    """About four times the distance to float64 that the operator shows: one
    rounding of each output (bf16 1.7e-3, fp16 2.1e-4, relative 2-norm) and fp32
    sums (2e-7; the two-phase schedule merges rounded partial results)."""
    c = case
    if c["kind"] == "model":
        return {"rel": 3e-2}
    many = 2.0 if c["kind"] == "two_phase" else 1.0
    return {"bf16": {"rel": 7e-3 * many}, "fp16": {"rel": 9e-4 * many}, "fp32": {"rel": 2e-6 * many}}[c["dtype"]]


def _attn_res(v, w):
    """``v [N, tokens, D]``, ``w [S, D]`` in float64 -> ``[S, tokens, D]``."""
    r = torch.rsqrt(v.square().mean(-1) + EPS)
    logits = (v @ w.T) * r.unsqueeze(-1)  # [N, tokens, S]
    a = torch.softmax(logits, dim=0).permute(2, 1, 0)  # [S, tokens, N]
    return torch.stack([(x.T.unsqueeze(-1) * v).sum(0) for x in a])


def exact(case, seed):
    c = case
    if c["kind"] == "model":
        return {"logits": _exact_model(c, seed)}
    x = _inputs(c, seed)
    n, d, tok = c["n"], c["d"], c["b"] * c["t"]
    v = x["v"].reshape(n, tok, d)
    s = c.get("s", 1)
    p = [x["w"].double().requires_grad_(c["grad"])]
    if c["kind"] == "module":
        p.append(x["gain"].double().requires_grad_(c["grad"]))
    g = x["g"].reshape(s, tok, d) if c["grad"] else None
    outs, dvs, dps = [], [], [torch.zeros_like(y) for y in p]
    step = max(1, min(tok, (1 << 25) // (n * d * s)))
    for t0 in range(0, tok, step):
        vv = v[:, t0 : t0 + step].double().requires_grad_(c["grad"])
        q = p[0] * p[1] if len(p) > 1 else p[0]
        o = _attn_res(vv, q.reshape(s, d))
        outs.append(o.detach())
        if c["grad"]:
            gv, *gp = torch.autograd.grad(o, [vv, *p], g[:, t0 : t0 + step].double())
            dvs.append(gv)
            dps = [a + b for a, b in zip(dps, gp)]
    shape = (c["b"], c["t"], d)
    out = torch.cat(outs, 1).reshape(*((s,) if c["kind"] == "batched" else ()), *shape)
    if not c["grad"]:
        return {"out": out}
    dv = torch.cat(dvs, 1).reshape(n, *shape)
    dp = [y.detach() for y in dps]
    return {"out": out, "grads": [*dv.unbind(0), *dp] if c["kind"] == "sources" else [dv, *dp]}


def _exact_model(c, seed):
    w, idx = _model_inputs(c, seed)
    w = {k: y.double() for k, y in w.items()}
    b, t, d, h = c["b"], c["t"], c["d"], c["heads"]
    hd, half = d // h, d // h // 2
    ang = (torch.arange(t, device=DEV, dtype=torch.float64)[:, None]
           * 10000.0 ** (-torch.arange(half, device=DEV, dtype=torch.float64) * 2.0 / hd)[None])
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    mask = torch.ones(t, t, device=DEV, dtype=torch.bool).triu(1)

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w[name]

    def turn(x):
        lo, hi = x.chunk(2, -1)
        return torch.cat((lo * cos - hi * sin, lo * sin + hi * cos), -1)

    def attention(x, i):
        q, k, v = (x @ w[f"layers.{i}.attn.qkv.weight"].T).view(b, t, 3, h, hd).unbind(2)
        q, k, v = (y.transpose(1, 2).contiguous() for y in (turn(q), turn(k), v))
        a = (q @ k.transpose(-1, -2).contiguous() / hd**0.5).masked_fill(mask, -math.inf).softmax(-1)
        return (a @ v).transpose(1, 2).reshape(b, t, d) @ w[f"layers.{i}.attn.out.weight"].T

    def mlp(x, i):
        a, u = (x @ w[f"layers.{i}.mlp.gate_up.weight"].T).chunk(2, -1)
        return (torch.nn.functional.silu(a) * u) @ w[f"layers.{i}.mlp.down.weight"].T

    def site(i, sources):
        q = w[f"attn_res.{i}.w"] * w[f"attn_res.{i}.g"]
        return _attn_res(torch.stack(sources).reshape(len(sources), b * t, d), q[None])[0].reshape(b, t, d)

    per = 2 * c["layers"] // c["blocks"]
    done, running = [w["embed.weight"][idx]], None
    for i in range(2 * c["layers"]):
        if i > 0 and i % per == 0:
            done, running = [*done, running], None
        x = site(i, done + ([running] if running is not None else []))
        y = attention(norm(x, f"layers.{i // 2}.attn_norm.weight"), i // 2) if i % 2 == 0 else mlp(
            norm(x, f"layers.{i // 2}.mlp_norm.weight"), i // 2)
        running = y if running is None else running + y
    x = site(2 * c["layers"], [*done, running])
    return norm(x, "final_norm.weight") @ w["lm_head.weight"].T
