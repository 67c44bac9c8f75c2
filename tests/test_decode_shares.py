"""Host test: how many stream-K shares a lone long sequence gets when the
merge takes up to 256 pieces of a segment (the backend's kernel fact), and
when the fact is left out (at most 48)."""

from __future__ import annotations

import pytest
import torch

import light_vllm_amd as lv
from light_vllm_amd.plan import DECODE_MERGE_PIECES, KERNEL_FACTS, StepPlan

# 4 kv heads, 16-token blocks, 1024 resident waves of 32-token tiles.
FACTS = (7, 4, 16, 0, 0, 0, 0, 0, 1, 0, 1024, 32, 0, 0, 0, 0, 0, 16, 1, 4, 0, 0, 0, 0, 8)


def _work(computed: int, *optional: int):
    md = lv.PagedAttentionMetadata(block_tables=(tuple(range(-(-(computed + 1) // 16))),),
                                   num_computed_tokens=(computed,), query_layouts=(lv.linear_query_layout(1),))
    return StepPlan(md, block_size=16, device=torch.device("cpu")).layer_work(FACTS + optional)


@pytest.mark.parametrize("tokens, shares", ((33, 2), (96 * 32, 96), (96 * 32 + 1, 49), (8112, 127), (256 * 32, 128),
                                            (512 * 32, 171), (32701, 205), (65536, 228)))
def test_lone_sequence_shares(tokens, shares) -> None:
    work = _work(tokens - 1, DECODE_MERGE_PIECES)
    assert work.waves_per_head == shares <= DECODE_MERGE_PIECES
    pieces = work.pieces.numpy()
    assert pieces[0][2] == 0 and pieces[-1][3] == tokens  # whole, in order, without gaps
    assert pieces[:-1, 3].tolist() == pieces[1:, 2].tolist()
    assert work.jobs.numpy()[0][3] == len(pieces) == work.num_partial_slots
    assert _work(tokens - 1).waves_per_head <= 48 or tokens > 48 * 254 * 16  # (long pieces are capped by their table)


def test_kernel_facts_may_leave_out_only_the_optional_ones() -> None:
    assert len(FACTS) + 1 == len(KERNEL_FACTS)
    assert _work(5000).pieces.tolist() == _work(5000, 0).pieces.tolist()
    with pytest.raises(ValueError):
        _work(5000, 0, 0)
