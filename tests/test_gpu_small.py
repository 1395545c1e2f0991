"""The small form (k_layer_small, k_experts_small: 2, 4 or 8 units per 128-row block of gate and up, at
up to 16 tokens): the single launch against the stream-ordered kernels, bit for bit, for each number of
parts the geometry allows, both activation forms, 0 to 2 shared experts, the dense schedule (with experts
the routing leaves unpicked) and the routed one, 2, 4 and 8 K parts of the down units; and both against
the CPU oracle."""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

import bench
from oracle import layer, metrics
from tests.down_parts import down_parts
from vibe_megakernel_amd import cases as C
from vibe_megakernel_amd import submission, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

MIXTRAL, DEEPSEEK, KIMI = "moe-fp8-mixtral-t16", "moe-fp8-deepseek-v3-t64", "moe-fp8-kimi-k2-t128"


def _case(base, act="fp8", **p):
    return replace(C.development(C.case(base), **p), activations=act)


def _cases():
    out = []
    for act in ("fp8", "bf16"):
        # Routed: 3, 2 and 4 or more K blocks a row allow 2, 4 and 8 parts.
        out += [_case(MIXTRAL, act, tokens=t, experts=64, hidden=h) for t, h in ((1, 384), (3, 256), (2, 512), (16, 1152))]
        out += [_case(DEEPSEEK, act, tokens=t, experts=64, shared_experts=s, intermediate=i)
                for t, s, i in ((1, 1, 128), (2, 1, 384), (5, 2, 256))]
        # Dense: blocks of 512 KB and more; 17, 18 and 20 K blocks allow 2, 4 and 8 parts.
        out += [_case(MIXTRAL, act, tokens=t, experts=8, hidden=h) for t, h in ((4, 2176), (5, 2304), (16, 2560))]
        out.append(_case(DEEPSEEK, act, tokens=15, experts=32, topk=4, hidden=2048, shared_experts=2))
        out.append(replace(_case(KIMI, act, tokens=12), norm="fp32_weight", residual=True))  # dense: whole blocks
        out.append(replace(_case(KIMI, act, tokens=12, experts=64), norm="fp32_weight", residual=True))
    for experts in (16, 64):  # dense: whole blocks; routed: parts
        out.append(replace(_case(DEEPSEEK, tokens=4, experts=experts), swiglu="bf16", swiglu_limit=0.5, power_of_two=True))
    return out


def _id(c):
    return (f"{c.model.split('/')[-1].split()[0]}-{c.activations}-t{c.tokens}-e{c.experts}-h{c.hidden}-i{c.intermediate}"
            f"-s{c.shared_experts}")


def _check(case):
    print(_id(case), flush=True)
    one, five = submission.MoELayer(case), submission.MoELayer(case, single_launch=False)
    for seed in (3, 4):  # consecutive calls on one workspace
        host = workloads.make_inputs(case, seed, "cpu")
        values = {k: v.to(DEV) for k, v in host.items()}
        a, b = one(values), five(values)
        torch.cuda.synchronize()
        assert not one.gave_up(torch.device(DEV))
        for k in ("y", "expert_ids", "expert_weights"):
            assert torch.equal(a[k], b[k]), k
    want = layer.block_reference(case, host) if case.residual else layer.reference(case, host)
    check = metrics.layer_checks(a["y"], want["y"])  # the layer's bars: max-rel 1e-2, cosine 0.9999
    assert torch.equal(a["expert_ids"].cpu(), want["expert_ids"]) and check["pass"], check
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        one(values)
        five(values)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events()]
    for kernel in (bench.layer_kernel(case), bench.expert_kernel(case)):
        assert ("_small<" in kernel) == (bench._parts(case) > 1) and any(f"::{kernel}(" in n or f" {kernel}(" in n
                                                                         for n in names), (kernel, names)


@pytest.mark.parametrize("case", _cases(), ids=_id)
def test_small_units_equal_the_stream_ordered_kernels_and_the_oracle(case):
    _check(case)


def test_the_cases_have_every_number_of_units_a_block():
    for act in ("fp8", "bf16"):
        for dense in (False, True):
            got = {bench._parts(c) for c in _cases() if c.activations == act and bench._dense(c) == dense}
            assert got >= {2, 4, 8}, (act, dense, got)


def _part_cases():
    # Down units of 2, 4 and 8 K parts under both schedules, with and without a shared expert.
    for act in ("fp8", "bf16"):
        for parts, intermediate in ((2, 2048), (4, 4096), (8, 8192)):
            yield parts, _case(MIXTRAL, act, tokens=1, experts=16, hidden=512, intermediate=intermediate)
            yield parts, _case(DEEPSEEK, act, tokens=2, experts=16, topk=2, hidden=512, intermediate=intermediate)
        yield 2, _case(DEEPSEEK, act, tokens=3, experts=16, topk=2, hidden=512, intermediate=2048, shared_experts=2)
        yield 2, _case(MIXTRAL, act, tokens=5, experts=4, hidden=2048, intermediate=2048)
        yield 4, _case(DEEPSEEK, act, tokens=9, experts=8, hidden=2048, intermediate=4096)


@pytest.mark.parametrize("parts,case", list(_part_cases()), ids=lambda v: _id(v) if isinstance(v, C.Case) else f"ks{v}")
def test_small_units_with_k_parts(parts, case):
    assert down_parts(case) == parts and bench._parts(case) > 1
    _check(case)


def test_small_kernel_is_one_launch():
    case = _case(DEEPSEEK, tokens=1)
    run = submission.MoELayer(case)
    values = {k: v.to(DEV) for k, v in workloads.make_inputs(case, 3, "cpu").items()}
    run(values)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        run(values)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "k_" in e.name]
    assert len(names) == 1 and "k_layer_small" in names[0], names
