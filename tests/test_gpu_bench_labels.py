"""bench.py names the kernel that runs: its labels against the profiler's kernel names, over a geometry
of every form and both sides of the lines between them."""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

import bench
from vibe_megakernel_amd import cases as C
from vibe_megakernel_amd import submission, workloads

DEV = "cuda:0"
MIXTRAL, QWEN, MX = "moe-fp8-mixtral-t16", "moe-fp8-qwen3-30b-a3b-t32", "moe-mxfp4-deepseek-v4-pro-t64"


def _case(base, act="fp8", **p):
    return replace(C.development(C.case(base), **p), activations=act)


def _cases():
    for act in ("fp8", "bf16"):
        yield _case(QWEN, act, tokens=1, experts=64, hidden=512)                      # 8 parts
        yield _case(MIXTRAL, act, tokens=16, experts=8, hidden=2048)                  # dense, parts
        yield _case(MIXTRAL, act, tokens=16, experts=8, hidden=256)                   # dense, whole blocks
        yield _case(MIXTRAL, act, tokens=40, experts=8, hidden=4096)                  # W8A8: gate and up apart
        yield _case(MIXTRAL, act, tokens=80, experts=8, hidden=4096)                  # 20 rows an expert
        yield _case(QWEN, act, tokens=207, experts=128, topk=8)
        yield _case(QWEN, act, tokens=208, experts=128, topk=8)
        yield _case(QWEN, act, tokens=208, experts=128, topk=7)
        yield _case(QWEN, act, tokens=449, experts=1024, topk=8)
        yield _case(MIXTRAL, act, tokens=143, experts=32, topk=1, hidden=4096, intermediate=2048)
        yield _case(MIXTRAL, act, tokens=144, experts=32, topk=1, hidden=4096, intermediate=2048)
        yield _case(MIXTRAL, act, tokens=144, experts=32, topk=1, hidden=4096, intermediate=1920)
    for tokens in (14, 16, 23, 24, 47, 48):  # of 4 experts, top-2
        yield _case(MX, tokens=tokens, experts=4, topk=2, hidden=2048, intermediate=4096)
        yield _case(MX, tokens=tokens, experts=4, topk=2, hidden=512, intermediate=4096)


def _id(c):
    return f"{c.format}-{c.activations}-t{c.tokens}-e{c.experts}-k{c.topk}-h{c.hidden}-i{c.intermediate}"


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(_cases()), ids=_id)
def test_labels_are_the_kernels_that_run(case):
    print(_id(case), flush=True)
    values = workloads.make_inputs(case, 3, DEV)
    for single, label in ((True, bench.layer_kernel(case)), (False, bench.expert_kernel(case))):
        run = submission.MoELayer(case, single_launch=single)
        run(values)
        torch.cuda.synchronize()
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            run(values)
            torch.cuda.synchronize()
        names = [e.name for e in prof.events()]
        assert any(f"::{label}(" in n or f" {label}(" in n for n in names), (label, names)


def test_labels_of_the_catalog():
    assert {c.id: bench.layer_kernel(c) for c in C.CASES} == {
        "moe-fp8-tiny-t4": "k_layer<false, false>",
        "moe-fp8-mixtral-t16": "k_layer_small<false>",
        "moe-fp8-qwen3-30b-a3b-t32": "k_layer<false, false>",
        "moe-fp8-deepseek-v3-t64": "k_layer<false, false>",
        "moe-fp8-kimi-k2-t128": "k_layer<false, false>",
    }
    assert bench.expert_kernel(C.case(MIXTRAL)) == "k_experts_small<false>"
    assert bench.layer_kernel(C.case(MX)) == "k_layer_mx" and bench.expert_kernel(C.case(MX)) == "k_experts_mx"
