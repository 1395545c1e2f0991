"""The number of K parts of a geometry's down units, from the library's workspace size."""

from __future__ import annotations

from dataclasses import replace

from vibe_megakernel_amd import submission


def down_parts(case) -> int:
    """Against one 128-column block of h less, whose odd number of K blocks leaves one part and no
    partial rows, the workspace grows by the fp32 partials [parts, rows, H] of the routed (dense
    schedule: every expert's) and shared rows, and by far less than one part's for the block itself."""
    T, H, E, K, I = case.tokens, case.hidden, case.experts, case.topk, case.intermediate
    assert I // 128 % 2 == 0
    rows = (E * T if T <= 16 and T * K >= E else T * K) + (T if case.shared_experts else 0)
    fewer = replace(case, params=dict(case.params, intermediate=I - 128))
    size = submission.MoELayer(case).workspace_bytes - submission.MoELayer(fewer).workspace_bytes
    return max(1, size // (4 * rows * H))
