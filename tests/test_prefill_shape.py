"""Host test: the workgroup shape a prefill step's plan takes (key tiles per
resident 8-wave workgroup; the mean per unit where units are not split)."""

from __future__ import annotations

import pytest
import torch

import light_vllm_amd as lv
from light_vllm_amd.plan import StepPlan


def _waves(computed: int, queries: int, requests: int, *, split: int = 1, built: int = 1, forced: int = 0) -> int:
    blocks = -(-(computed + queries) // 16)
    md = lv.PagedAttentionMetadata(
        block_tables=tuple(tuple(range(r * blocks, (r + 1) * blocks)) for r in range(requests)),
        num_computed_tokens=(computed,) * requests, query_layouts=(lv.linear_query_layout(queries),) * requests)
    facts = (7, 4, 16, 128, 64, split, 0, forced, 1, built, 1024, 32, 0, 0, 512, 512, 0, 16, 1, 4, 0, 0, 0, 0, 8)
    return StepPlan(md, block_size=16, device=torch.device("cpu")).layer_work(facts).prefill_waves


# 128 slots per kv head: the line is 1,024 key tiles per head (128 columns of
# group 7 are 18 queries).
@pytest.mark.parametrize("computed,queries,requests,waves", (
    (0, 17, 1, 8), (64 * 1022, 18, 1, 8), (64 * 1023, 18, 1, 4), (0, 512, 7, 8), (0, 512, 8, 4), (14336, 2048, 1, 4)))
def test_shape_follows_the_tiles_per_slot(computed, queries, requests, waves) -> None:
    assert _waves(computed, queries, requests) == waves
    assert _waves(computed, queries, requests, built=0) == 4
    assert _waves(computed, queries, requests, forced=12 - waves) == 12 - waves


def test_without_split_the_mean_unit_decides() -> None:
    assert _waves(0, 512, 40, split=0) == 8 and _waves(3072, 512, 1, split=0) == 4
