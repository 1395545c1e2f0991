"""The decode units' sums keep their order: the outputs' bytes for inputs made on the CPU, against
digests recorded when the units of a geometry without a batch form started at K blocks by unit, and up to
16 tokens ran as whole blocks. A change of the order (rotations, K parts) is within the layer's bars and
shows only here."""

from __future__ import annotations

import hashlib
import json
from dataclasses import replace
from pathlib import Path

import pytest
import torch

import bench
from vibe_megakernel_amd import cases as C
from vibe_megakernel_amd import submission, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GOLDEN = json.loads((Path(__file__).parent / "golden" / "decode_bits.json").read_text())


def _cases():
    # 128 experts of 16 row blocks: no K parts; h of 2 and 3 K blocks, x of 16.
    qwen, deepseek = C.case("moe-fp8-qwen3-30b-a3b-t32"), C.case("moe-fp8-deepseek-v3-t64")
    for act in ("fp8", "bf16"):
        yield replace(C.development(qwen, tokens=40, hidden=2048, experts=128, topk=8, intermediate=256), activations=act)
        yield replace(C.development(deepseek, tokens=70, hidden=2048, experts=128, topk=4, intermediate=384), activations=act)
    # The small form with two units a block, dense and routed: whole-block units before it.
    mixtral = C.case("moe-fp8-mixtral-t16")
    for act in ("fp8", "bf16"):
        yield replace(C.development(mixtral, tokens=5, hidden=2176, experts=8, topk=2, intermediate=384), activations=act)
        yield replace(C.development(deepseek, tokens=3, hidden=1152, experts=64, topk=4, intermediate=384), activations=act)


def _id(c):
    return f"{c.activations}-t{c.tokens}-e{c.experts}-h{c.hidden}-i{c.intermediate}-s{c.shared_experts}"


def digest(case, single_launch):
    values = workloads.make_inputs(case, 17, "cpu")
    run = submission.MoELayer(case, single_launch=single_launch)
    y = run({k: v.to(DEV) for k, v in values.items()})["y"]
    torch.cuda.synchronize()
    return hashlib.sha256(y.cpu().view(torch.int16).numpy().tobytes()).hexdigest()


@pytest.mark.parametrize("single_launch", [True, False])
@pytest.mark.parametrize("case", list(_cases()), ids=_id)
def test_decode_units_keep_their_bits(case, single_launch):
    print(_id(case), flush=True)
    assert bench._parts(case) == (2 if case.tokens <= 16 else 1)
    assert digest(case, single_launch) == GOLDEN[_id(case)]
