"""The MXFP4 batch units (k_experts_mx_batch) at the edges of their chunk forms (rows of an expert up to
32, 64, 96 and 128, and several chunks an expert) against the decode units, which work the same rows in
calls of fewer rows: bit for bit, the order of a row's sums being the geometry's alone."""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

from vibe_megakernel_amd import cases as C
from vibe_megakernel_amd import ep as EP
from vibe_megakernel_amd import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPCASE = C.case("megamoe-layer-deepseek-v4-pro-ep8-t512")
LOCAL = 4


@pytest.mark.parametrize("hidden,intermediate", [(512, 4096), (1024, 4096)])
@pytest.mark.parametrize("counts", [(32, 33, 31, 1), (64, 65, 63, 0), (96, 97, 95, 17), (128, 129, 127, 16),
                                    (300, 2, 192, 225), (0, 0, 0, 100)])
def test_chunk_edges_equal_small_calls(counts, hidden, intermediate):
    print(counts, hidden, intermediate, flush=True)
    R = sum(counts)
    case = replace(EPCASE, id="mx-chunks", gpus=1, ep=1,
                   params=dict(tokens=R, experts=LOCAL, topk=1, hidden=hidden, intermediate=intermediate))
    v = {k: t.to(DEV) for k, t in workloads.make_mx_inputs(workloads.serial_case(case), 31).items()}
    ids = torch.repeat_interleave(torch.arange(LOCAL), torch.tensor(counts))
    ids = ids[torch.randperm(R, generator=torch.Generator().manual_seed(5))].to(DEV)
    experts = EP.Experts(v["l1_blocks"], v["l1_scales"], v["l2_blocks"], v["l2_scales"], 0, case.swiglu_limit)
    args = (v["x"], v["x_scales"], ids, v["topk_weights"].flatten())
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        got = experts(*args)
        torch.cuda.synchronize()
    assert any("k_experts_mx_batch" in e.name for e in prof.events())
    step = 24 * LOCAL - 4  # decode units: fewer than 24 rows an expert on average
    for r in range(0, R, step):
        part = [a[max(0, min(r, R - step)):][:step].contiguous() for a in args]  # as many rows: the same K parts
        want = experts(*part)
        torch.cuda.synchronize()
        assert torch.equal(got[max(0, min(r, R - step)):][:step], want), r


@pytest.mark.parametrize("local,rows,batch", [(64, 8, True), (72, 12, False), (72, 13, True)])
def test_many_experts_keep_the_decode_units_longer(local, rows, batch):
    """Large experts (8M weights a matrix): 64 of them take the batch units from 8 rows an expert, more
    of them from 13; the same bits as in calls of fewer rows."""
    print(local, rows, flush=True)
    case = replace(EPCASE, id="mx-many", gpus=1, ep=1,
                   params=dict(tokens=local * rows, experts=local, topk=1, hidden=4096, intermediate=2048))
    v = {k: t.to(DEV) for k, t in workloads.make_mx_inputs(workloads.serial_case(case), 31, DEV).items()}
    ids = (torch.arange(local * rows) % local).to(DEV)
    experts = EP.Experts(v["l1_blocks"], v["l1_scales"], v["l2_blocks"], v["l2_scales"], 0, case.swiglu_limit)
    args = (v["x"], v["x_scales"], ids, v["topk_weights"].flatten())
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        got = experts(*args)
        torch.cuda.synchronize()
    assert any("k_experts_mx_batch" in e.name for e in prof.events()) == batch
    step = 4 * local  # decode units
    for r in range(0, local * rows - step + 1, step):
        want = experts(*[a[r:r + step].contiguous() for a in args])
        torch.cuda.synchronize()
        assert torch.equal(got[r:r + step], want), r
