"""Performance cases: the mixture-of-experts layer calls a serving program makes.

A program that serves one of the models of ``vibe_megakernel_amd.cases`` builds the layer once
(``submission.build``), keeps the weights on the GPU and calls ``run(inputs)`` for every layer
of every step. What varies in use is the number of tokens in the step (one user decoding, a
decode batch of any size, a chunk of a prompt), the model's geometry and routing, the numeric
form (W8A8, W8A16, power-of-two scales, MXFP4) and whether the layer runs alone or as the
decoder block's MoE half (RMSNorm before, residual after). Under expert parallelism a rank
calls ``ep.dispatch``, its local experts and ``ep.combine`` around the program's own
exchanges. The listed cases cover that range; ``draw`` takes other points of it.
"""

from __future__ import annotations

import importlib
import math
from dataclasses import replace

import torch

import __graft_entry__

__graft_entry__.load_package()  # the package directory's name is not an identifier
catalog = importlib.import_module("vibe_megakernel_amd.cases")
workloads = importlib.import_module("vibe_megakernel_amd.workloads")
submission = importlib.import_module("vibe_megakernel_amd.submission")
ep = importlib.import_module("vibe_megakernel_amd.ep")

DEVICE = "cuda:0"

# The catalog's geometries; `most`: the largest token count drawn.
FAMILIES = {
    "tiny": ("moe-fp8-tiny-t4", 64),
    "mixtral": ("moe-fp8-mixtral-t16", 512),
    "qwen3": ("moe-fp8-qwen3-30b-a3b-t32", 2048),
    "glm": ("moe-fp8-glm-5.3-flash-t64", 512),
    "deepseek": ("moe-fp8-deepseek-v3-t64", 512),
    "kimi": ("moe-fp8-kimi-k2-t128", 128),
    "deepseek-mx": ("moe-mxfp4-deepseek-v4-pro-t64", 256),
    "deepseek-ep": ("megamoe-layer-deepseek-v4-pro-ep8-t512", 512),
}


def _case(family, tokens, name=None, activations="fp8", pow2=False, block=False, bias_std=0.1):
    c = {"family": family, "tokens": tokens, "activations": activations, "pow2": pow2, "block": block,
         "bias_std": bias_std}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # One user decoding: a handful of experts, so launches and the routing's latency count.
        _case("qwen3", 1, "qwen3-t1"),
        # The same on a large model, in the numerics and the block form its decoder runs.
        _case("deepseek", 1, "deepseek-t1-w8a16-block", activations="bf16", pow2=True, block=True),
        # A few users on a model of few, wide experts (every expert is likely hit).
        _case("mixtral", 5, "mixtral-t5"),
        # An ordinary decode batch of a small model, as its decoder block.
        _case("qwen3", 32, "qwen3-t32-block", block=True),
        # A decode batch of no round size; clamped SwiGLU.
        _case("glm", 37, "glm-t37"),
        # The benchmark's shape.
        _case("deepseek", 64, "deepseek-t64"),
        # A larger decode batch under skewed routing: a few hot experts, most of them hit.
        _case("kimi", 128, "kimi-t128"),
        # bf16 activations at a large decode batch.
        _case("deepseek", 256, "deepseek-t256-w8a16", activations="bf16", pow2=True),
        # The largest decode batch of a rank (and a short prompt chunk).
        _case("deepseek", 512, "deepseek-t512"),
        # A chunk of a prompt (prefill).
        _case("qwen3", 2000, "qwen3-t2000"),
        # MXFP4 experts at a decode batch (routing given).
        _case("deepseek-mx", 64, "deepseek-mx-t64"),
        # One rank's share of the expert-parallel layer at its catalog size.
        _case("deepseek-ep", 512, "deepseek-ep8-t512"),
    ]


def draw(rng):
    while True:
        family = rng.choice(("tiny", "mixtral", "qwen3", "qwen3", "glm", "deepseek", "deepseek", "kimi",
                             "deepseek-mx", "deepseek-ep"))
        tokens = int(round(math.exp(rng.uniform(0.0, math.log(FAMILIES[family][1])))))
        c = _case(family, tokens)
        if family == "deepseek-ep":  # decode batches per rank
            c["tokens"] = int(round(math.exp(rng.uniform(math.log(16), math.log(512)))))
        elif family != "deepseek-mx":
            c["block"] = rng.random() < 0.5
            if family in ("deepseek", "kimi"):  # the DeepSeek family's forms
                c["activations"] = rng.choice(("fp8", "fp8", "bf16"))
                c["pow2"] = rng.random() < 0.5
                c["bias_std"] = rng.choice((0.03, 0.1))  # how evenly the correction bias spreads the experts
                if c["activations"] == "bf16":  # costs more per token past the listed size
                    c["tokens"] = min(c["tokens"], 256)
        if all(any(c[key] != l[key] for key in c) for l in listed()):
            return c


def _layer_case(c):
    """The catalog's record with this case's tokens and form."""
    k = catalog.case(FAMILIES[c["family"]][0])
    k = replace(k, id="perf", params=dict(k.params, tokens=c["tokens"]))
    if c["family"] in ("deepseek-mx", "deepseek-ep"):
        return k
    k = replace(k, activations=c["activations"], power_of_two=c["pow2"], bias_std=c["bias_std"])
    if c["block"]:  # gamma in fp32 for the DeepSeek family, on the rounded row otherwise
        sigmoid = k.router == "sigmoid"
        k = replace(k, norm="fp32_weight" if sigmoid else "bf16_weight", norm_eps=1e-6 if sigmoid else 1e-5,
                    residual=True)
    return k


def _inputs(c, seed):
    k = _layer_case(c)
    if k.ep == 1:
        return workloads.make_inputs(k, seed, DEVICE)
    # Rank 0's share: its own tokens, and the rows every rank sends it (in the order the
    # exchange delivers them: by source rank, then token and slot), cut or filled up from the
    # first ones to the average count T*K, so that every seed has as many.
    v = workloads.make_ep_inputs(k, seed, DEVICE, rank=0)
    ids = v["topk_idx"].flatten()
    got = (ids < k.experts // k.ep).nonzero().flatten()
    got = got[torch.arange(k.tokens * k.topk, device=DEVICE) % got.numel()]
    source = got // k.topk
    gen = torch.Generator(device=DEVICE).manual_seed(workloads.seed_for(seed, "returned"))
    back = torch.randn((k.tokens * k.topk, k.hidden), generator=gen, device=DEVICE)
    own = slice(0, k.tokens)
    return {"x": v["x"][own].contiguous(), "x_scales": v["x_scales"][own].contiguous(),
            "topk_idx": v["topk_idx"][own].contiguous(), "topk_weights": v["topk_weights"][own].contiguous(),
            "rows": v["x"].view(torch.uint8)[source].view(torch.float8_e4m3fn), "row_scales": v["x_scales"][source],
            "row_ids": ids[got].contiguous(), "row_weights": v["topk_weights"].flatten()[got].contiguous(),
            "returned": back.to(torch.bfloat16),
            **{n: v[n] for n in ("l1_blocks", "l1_scales", "l2_blocks", "l2_scales")}}


def prepare(case, seed):
    k = _layer_case(case)
    v = _inputs(case, seed)
    if k.ep == 1:
        return {"run": submission.build(k.to_dict()), "inputs": v}
    experts = ep.Experts(v["l1_blocks"], v["l1_scales"], v["l2_blocks"], v["l2_scales"], 0, k.swiglu_limit)
    rows = v["rows"].shape[0]
    return {"ep": k.ep, "experts": k.experts, "inputs": v, "local": experts,
            "workspace": torch.empty(experts.workspace_bytes(rows), dtype=torch.uint8, device=DEVICE)}


def run(state):
    v = state["inputs"]
    if "run" in state:
        return state["run"](v)
    # The rank's three steps around the program's two exchanges (whose results are inputs).
    send = ep.dispatch(v["x"], v["x_scales"], v["topk_idx"], v["topk_weights"], state["experts"], state["ep"])
    out = state["local"](v["rows"], v["row_scales"], v["row_ids"], v["row_weights"], workspace=state["workspace"])
    y = ep.combine(v["returned"], send.slot_rows)
    return {"rows": send.rows.view(torch.uint8), "row_scales": send.row_scales, "ids": send.ids,
            "weights": send.weights, "counts": send.counts, "slot_rows": send.slot_rows, "out": out, "y": y}


def _hit(k):
    """Experts hit by the routing of a call, on average: the selection rule over logits with the
    inputs' distribution (independent normals of the router's spread)."""
    gen = torch.Generator().manual_seed(5)
    hits = []
    for s in range(3):
        if k.router == "given":
            tokens = k.tokens * k.ep
            pop = torch.randn(k.experts, generator=gen) * 0.4
            score = pop - torch.log(-torch.log(torch.rand((tokens, k.experts), generator=gen).clamp(1e-12, 1 - 1e-7)))
            ids = score.topk(k.topk, -1).indices
            hits.append(int((ids.unique() < k.experts // k.ep).sum()))
            continue
        logits = torch.randn((k.tokens, k.experts), generator=gen) * (k.router_std * k.hidden ** 0.5)
        bias = workloads.router_bias(k, 100 + s, "cpu")
        hits.append(len(_route(k, logits.double(), None if bias is None else bias.double())[0].unique()))
    return sum(hits) / len(hits)


def work(case):
    k = _layer_case(case)
    T, H, E, K, I, S = k.tokens, k.hidden, k.experts, k.topk, k.intermediate, k.shared_experts
    hit = _hit(k)
    if k.ep > 1:
        n, rows = T * K, T * K  # rows sent and received
        weights = hit * (3 * I * H // 2 + 3 * I * H // 32)
        row = H + H // 32 + 12
        return {"bytes": weights + T * (H + H // 32) + 12 * n + n * (row + 4)  # dispatch
                + rows * row + 2 * rows * H                                      # local experts
                + 2 * n * H + 4 * n + 2 * T * H,                                  # combine
                "flops": 6 * rows * H * I + n * H}
    if k.format == "mxfp4":
        return {"bytes": hit * (3 * I * H // 2 + 3 * I * H // 32) + T * (H + H // 32) + 12 * T * K + 2 * T * H,
                "flops": 6 * T * K * H * I}
    per = 3 * I * H + 4 * 3 * (I // 128) * (H // 128)
    return {"bytes": (hit + S) * per + 4 * E * H + (4 * E if k.bias != "none" else 0)
            + (2 * H if k.norm != "none" else 0) + 4 * T * H + 12 * T * K,
            "flops": 2 * T * E * H + 6 * T * (K + S) * H * I}


def tolerance(case):
    # Against the 64-bit sums below, with the format's own roundings kept, y is within 1.7e-3
    # (the rounding of y to bf16 alone) to 3.1e-3 (a sum near a rounding boundary of bf16, and
    # from there of E4M3, takes the other neighbour) over listed and drawn cases, the weights
    # of the routing within 5e-6; the ids are exact.
    return {"rel": 1e-2, "differ": 1e-3}


# -- the same layer in 64 bits ----------------------------------------------------------------


def _bf16(v):
    return v.to(torch.bfloat16).double()


def _route(k, logits, bias):
    """ids [T, K] and weights of fp64 logits: stable descending order, lower index first."""
    if k.router == "softmax":
        ids = logits.argsort(dim=-1, descending=True, stable=True)[:, :k.topk]
        return ids, logits.gather(1, ids).softmax(-1) * k.routed_scaling
    prob = logits.sigmoid()
    choice = prob if bias is None else prob + bias
    if k.groups > 1:
        groups = choice.unflatten(-1, (k.groups, -1))
        score = groups.topk(2, -1).values.sum(-1)
        keep = score.argsort(dim=-1, descending=True, stable=True)[:, :k.top_groups]
        drop = torch.ones_like(score, dtype=torch.bool).scatter_(1, keep, False)
        choice = groups.masked_fill(drop[..., None], -math.inf).flatten(1)
    ids = choice.argsort(dim=-1, descending=True, stable=True)[:, :k.topk]
    w = prob.gather(1, ids)
    return ids, w / (w.sum(-1, keepdim=True) + 1e-20) * k.routed_scaling


def _e4m3_128(v, pow2):
    """bf16-valued rows through E4M3 with one fp32 scale per 128."""
    g = v.float().unflatten(-1, (-1, 128))
    amax = g.abs().amax(-1, keepdim=True).clamp_min(1e-4)
    s = amax / torch.full_like(amax, 448.0)  # the fp32 quotient (by a scalar torch takes its reciprocal)
    if pow2:
        s = torch.exp2(torch.ceil(torch.log2(s)))
    return ((g / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double() * s.double()).flatten(-2)


def _weight(q, s):
    r, c = q.shape
    return (q.double().view(r // 128, 128, c // 128, 128) * s.double()[:, None, :, None]).view(r, c)


def _mlp(k, x, gate, up, down):
    quant = (lambda v: _e4m3_128(v, k.power_of_two)) if k.activations == "fp8" else (lambda v: v)
    xq = quant(x)
    g, u = _bf16(xq @ _weight(*gate).T), _bf16(xq @ _weight(*up).T)
    if k.swiglu_limit > 0:
        g, u = g.clamp(max=k.swiglu_limit), u.clamp(-k.swiglu_limit, k.swiglu_limit)
    s = g * g.sigmoid()
    h = _bf16((_bf16(s) if k.swiglu == "bf16" else s) * u)
    return _bf16(quant(h) @ _weight(*down).T)


def _exact_layer(k, v):
    x = v["x"].double()
    if k.norm != "none":
        n = x / (x.square().mean(-1, keepdim=True) + k.norm_eps).sqrt()
        x = _bf16((n if k.norm == "fp32_weight" else _bf16(n)) * v["ln2"].double())
    bias = v["router_bias"].double() if k.bias != "none" else None
    ids, w = _route(k, (x @ v["router"].double().T).float().double(), bias)
    pair = lambda name, e: (v[name][e], v[name + "_scale"][e])  # noqa: E731
    y = torch.zeros_like(x)
    for e in ids.unique().tolist():
        t, slot = (ids == e).nonzero(as_tuple=True)
        y[t] += _mlp(k, x[t], pair("gate", e), pair("up", e), pair("down", e)) * w[t, slot][:, None]
    if k.shared_experts:
        y += _mlp(k, x, *((v["shared_" + n], v[f"shared_{n}_scale"]) for n in ("gate", "up", "down")))
    if k.residual:
        y = v["x"].double() + _bf16(y)
    return {"y": y, "expert_ids": ids, "expert_weights": w}


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _mxfp4(blocks, scales):
    lut = torch.tensor(_E2M1, dtype=torch.float64, device=blocks.device)
    codes = torch.stack((blocks & 15, blocks >> 4), -1).flatten(-2).int()
    return (lut[codes] * torch.exp2(scales.double() - 127.0)[..., None]).flatten(-2)


def _e4m3_32(payload, scales):
    return (payload.double().unflatten(-1, (-1, 32)) * torch.exp2(scales.double() - 127.0)[..., None]).flatten(-2)


def _requant_32(a):
    """fp32 rows through E4M3 with E8M0 scales per 32: 2^(e-127) the smallest power of two with
    amax / 2^(e-127) <= 448, e at least 105."""
    g = a.float().unflatten(-1, (-1, 32))
    m, p = torch.frexp(g.abs().amax(-1).double())  # amax = m * 2^p, m in [0.5, 1)
    e = (p - 1 - 8 + (m * 2 > 1.75).to(p.dtype) + 127).clamp_min(105)
    s = torch.exp2(e.double() - 127.0)[..., None]
    return ((g.double() / s).float().to(torch.float8_e4m3fn).double() * s).flatten(-2)


def _exact_mx_rows(k, v, rows, ids, weights, base):
    """bf16-valued d of every row (its weight applied inside the SwiGLU)."""
    d = torch.zeros((rows.shape[0], k.hidden), dtype=torch.float64, device=rows.device)
    for e in ids.unique().tolist():
        at = (ids == e).nonzero().flatten()
        l1 = _bf16(rows[at] @ _mxfp4(v["l1_blocks"][e - base], v["l1_scales"][e - base]).T)
        gate, up = l1.chunk(2, -1)
        gate, up = gate.clamp(max=k.swiglu_limit), up.clamp(-k.swiglu_limit, k.swiglu_limit)
        h = _requant_32(gate * gate.sigmoid() * up * weights[at].double()[:, None])
        d[at] = _bf16(h @ _mxfp4(v["l2_blocks"][e - base], v["l2_scales"][e - base]).T)
    return d


def exact(case, seed):
    k = _layer_case(case)
    v = _inputs(case, seed)
    if k.format == "fp8":
        return _exact_layer(k, v)
    if k.ep == 1:
        rows = _e4m3_32(v["x"], v["x_scales"]).repeat_interleave(k.topk, 0)
        d = _exact_mx_rows(k, v, rows, v["topk_idx"].flatten(), v["topk_weights"].flatten(), 0)
        return {"y": d.view(k.tokens, k.topk, -1).sum(1)}
    ids = v["topk_idx"].flatten()
    owner = ids // (k.experts // k.ep)
    order = owner.argsort(stable=True)
    slot_rows = torch.empty_like(order)
    slot_rows[order] = torch.arange(order.numel(), device=order.device)
    source = order // k.topk
    out = _exact_mx_rows(k, v, _e4m3_32(v["rows"], v["row_scales"]), v["row_ids"], v["row_weights"], 0)
    return {"rows": v["x"].view(torch.uint8)[source], "row_scales": v["x_scales"][source], "ids": ids[order],
            "weights": v["topk_weights"].flatten()[order], "counts": owner.bincount(minlength=k.ep),
            "slot_rows": slot_rows.view(k.tokens, k.topk).int(), "out": out,
            "y": v["returned"].double()[slot_rows].view(k.tokens, k.topk, -1).sum(1)}
