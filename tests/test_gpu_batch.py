"""The single launch's batch units (k_layer_batch) against the stream-ordered kernels, whose decode
units compute the same sums: bit for bit at chunk sizes around the units' tiles (32, 64 and 128
rows and their remainders, more than one chunk an expert, experts no token picks), for both
activation forms, with a shared expert of several chunks, 2, 4 and 8 K parts of the down units and
the block steps; and against the CPU oracle once per form."""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

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
        # Every token picks both experts: each holds `tokens` rows.
        out += [_case(MIXTRAL, act, tokens=t, experts=2, topk=2) for t in (17, 32, 33, 64, 65, 96, 128, 129, 257)]
        # Ragged rows per expert; one K block a row of h; an odd number of K blocks; rows of H = 4096
        # (W8A8: gate and up apart, in both forms).
        out.append(_case(MIXTRAL, act, tokens=200, experts=8, intermediate=128))
        out.append(_case(MIXTRAL, act, tokens=300, experts=16, topk=3, hidden=768, intermediate=384))
        out.append(_case(MIXTRAL, act, tokens=70, experts=8, hidden=4096, intermediate=512))
        out.append(_case(DEEPSEEK, act, tokens=261))
        out.append(_case(KIMI, act, tokens=213, experts=16, topk=12))  # more slots than a load round of eight
        out.append(replace(_case(DEEPSEEK, act, tokens=300, shared_experts=2), norm="fp32_weight", residual=True))
        out.append(_case(KIMI, act, tokens=500, experts=32, topk=2))  # skewed: most experts hold few rows, some none
    out.append(replace(_case(DEEPSEEK, tokens=270), swiglu="bf16", swiglu_limit=0.5, power_of_two=True))
    return out


def _id(c):
    return f"{c.model.split('/')[-1].split()[0]}-{c.activations}-t{c.tokens}-e{c.experts}-h{c.hidden}-i{c.intermediate}"


def _equal_to_stream_ordered(case, kernel="k_layer_batch"):
    print(_id(case), flush=True)
    one, five = submission.MoELayer(case), submission.MoELayer(case, single_launch=False)
    for seed in (3, 4):  # consecutive calls on one workspace
        values = {k: v.to(DEV) for k, v in workloads.make_inputs(case, seed, "cpu").items()}
        a, b = one(values), five(values)
        torch.cuda.synchronize()
        assert not one.gave_up(torch.device(DEV))
        for k in ("y", "expert_ids", "expert_weights"):
            assert torch.equal(a[k], b[k]), k
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        one(values)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "k_" in e.name]
    assert len(names) == 1 and kernel in names[0], names
    return {k: v.cpu() for k, v in values.items()}, a


@pytest.mark.parametrize("case", _cases(), ids=_id)
def test_batch_units_equal_the_stream_ordered_kernels(case):
    _equal_to_stream_ordered(case, "k_layer<true" if case.activations == "fp8" and case.hidden == 4096 else "k_layer_batch")


def _part_cases():
    # 16, 32 and 64 K blocks a row of h: 2, 4 and 8 parts of eight. Chunks of up to 32, 64 and 128 rows
    # and more than one; a shared expert (parts of its own h rows, S*I wide), twice as wide in the last.
    for act in ("fp8", "bf16"):
        for parts, intermediate in ((2, 2048), (4, 4096), (8, 8192)):
            yield parts, _case(MIXTRAL, act, tokens=20, experts=2, topk=2, intermediate=intermediate)
            yield parts, _case(MIXTRAL, act, tokens=131, experts=4, topk=2, hidden=512, intermediate=intermediate)
            yield parts, _case(DEEPSEEK, act, tokens=70, experts=8, hidden=512, intermediate=intermediate)
        yield 2, replace(_case(DEEPSEEK, act, tokens=40, experts=8, intermediate=2048, shared_experts=2),
                         norm="fp32_weight", residual=True)


@pytest.mark.parametrize("parts,case", list(_part_cases()), ids=lambda v: _id(v) if isinstance(v, C.Case) else f"ks{v}")
def test_batch_units_with_k_parts(parts, case):
    assert down_parts(case) == parts
    host, got = _equal_to_stream_ordered(case)
    if case.tokens == 20:
        check = metrics.layer_checks(got["y"], layer.reference(case, host)["y"])  # max-rel 1e-2, cosine 0.9999
        assert check["pass"], check


def _few(tokens, experts, topk, batch, hidden=256, intermediate=256, act="fp8"):
    return _case(MIXTRAL, act, tokens=tokens, experts=experts, topk=topk, hidden=hidden, intermediate=intermediate), batch


@pytest.mark.parametrize("case,batch", [
    # Both sides of each line: 12 rows from 208 tokens, 3 up to 64 experts, 8 from 512 tokens, 2 from
    # 1024 and where the permute ranks in tiles (1024 experts from 449 tokens).
    _few(208, 512, 1, False), _few(208, 512, 1, False, act="bf16"), _few(208, 128, 7, False), _few(208, 128, 8, True),
    _few(207, 128, 8, False), _few(207, 64, 1, False), _few(208, 64, 1, True), _few(511, 128, 2, False),
    _few(512, 128, 2, True), _few(1023, 256, 2, False), _few(1024, 256, 2, True), _few(448, 1024, 8, False),
    _few(449, 1024, 8, True), _few(449, 1024, 4, False),
    # Experts of 8M weights: 4.5 rows from 128 tokens, 2 from 512.
    _few(128, 32, 1, False, 4096, 2048), _few(128, 32, 1, False, 4096, 2048, "bf16"), _few(143, 32, 1, False, 4096, 2048),
    _few(144, 32, 1, True, 4096, 2048), _few(144, 32, 1, True, 4096, 2048, "bf16"),
    _few(127, 16, 1, False, 2048, 4096), _few(128, 16, 1, True, 2048, 4096), _few(512, 256, 1, True, 8192, 1024),
    _few(512, 257, 1, False, 8192, 1024),
], ids=lambda v: f"t{v.tokens}-e{v.experts}-k{v.topk}-h{v.hidden}-{v.activations}" if isinstance(v, C.Case) else str(v))
def test_each_side_of_the_batch_line(case, batch):
    print(_id(case), flush=True)
    one, five = submission.MoELayer(case), submission.MoELayer(case, single_launch=False)
    values = workloads.make_inputs(case, 3, DEV)
    one(values)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        a = one(values)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "k_" in e.name]
    assert len(names) == 1 and ("k_layer_batch" in names[0]) == batch, names
    b = five(values)
    torch.cuda.synchronize()
    for k in ("y", "expert_ids", "expert_weights"):
        assert torch.equal(a[k], b[k]), k


def test_batch_kernel_runs_and_is_one_launch():
    case = _case(DEEPSEEK, tokens=256)
    run = submission.MoELayer(case)
    values = {k: v.to(DEV) for k, v in workloads.make_inputs(case, 3, "cpu").items()}
    run(values)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        run(values)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "k_" in e.name]
    assert len(names) == 1 and "k_layer_batch" in names[0], names


@pytest.mark.parametrize("act", ["fp8", "bf16"])
def test_batch_units_against_the_oracle(act):
    case = _case(MIXTRAL, act, tokens=150, experts=4)
    values = workloads.make_inputs(case, 11, "cpu")
    want = layer.reference(case, values)
    got = submission.MoELayer(case)({k: v.to(DEV) for k, v in values.items()})
    torch.cuda.synchronize()
    assert torch.equal(got["expert_ids"].cpu(), want["expert_ids"])
    check = metrics.layer_checks(got["y"], want["y"])  # the layer's bars: max-rel 1e-2, cosine 0.9999
    assert check["pass"], check
