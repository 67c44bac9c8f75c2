"""Host test: how many stream-K shares a lone long sequence gets when the
merge takes up to 256 pieces of a segment (the backend's kernel fact), and
when the fact is left out (at most 48)."""

from __future__ import annotations

import pytest
import torch

import light_vllm_amd as lv
from light_vllm_amd import native
from light_vllm_amd.plan import DECODE_MERGE_PIECES, KERNEL_FACTS, LayerShapes, StepPlan

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


# (lengths, bound on the merge's rounds of its deepest job): one deep segment
# beside many shallow ones, where the mean says nothing about the deepest.
@pytest.mark.parametrize("lens, rounds", (
    ([32702] + [300] * 63, 3), ([32702] + [300] * 31, 1), ([32702] * 2 + [400] * 30, 1), ([4000] + [200] * 31, 1),
    ([8111] + [64] * 31, 1), ([16000] + [1000] * 127, 4), ([65536], 1), ([1500] * 64, 1), ([300], 1)))
def test_merge_rounds_follow_the_deepest_job(lens, rounds) -> None:
    blocks = [-(-n // 16) for n in lens]
    tables = tuple(tuple(range(sum(blocks[:i]), sum(blocks[:i + 1]))) for i in range(len(lens)))
    md = lv.PagedAttentionMetadata(block_tables=tables, num_computed_tokens=tuple(n - 1 for n in lens),
                                   query_layouts=(lv.linear_query_layout(1),) * len(lens))
    key = FACTS + (DECODE_MERGE_PIECES,)
    plan = lambda **kw: StepPlan(md, block_size=16, device=torch.device("cpu"), **kw).layer_work(key)  # noqa: E731
    work, fused = plan(), plan(num_blocks=sum(blocks), shapes=LayerShapes([key]))
    depth = int(work.jobs.numpy()[:, 3].max())
    assert work.merge_depth == fused.merge_depth == depth <= DECODE_MERGE_PIECES
    waves = native.load().lvamd_paged_merge_waves(2, 128, work.num_jobs, work.num_partial_slots, depth, 4,
                                                  work.merge_columns)
    assert waves in (1, 4, 16) and -(-depth // (16 * waves)) <= rounds


def test_merge_waves_by_depth_mean_and_columns() -> None:
    waves = lambda jobs, partials, depth, heads=4, columns=7, d=128: (  # noqa: E731
        native.load().lvamd_paged_merge_waves(2, d, jobs, partials, depth, heads, columns))
    assert [waves(64, 312, n) for n in (9, 16, 17, 64, 65, 256)] == [1, 1, 4, 4, 4, 4]
    assert [waves(32, 200, n) for n in (16, 17, 64, 65, 256)] == [1, 4, 4, 16, 16]  # 256 workgroups of two per head
    assert [waves(32, n, 0) for n in (256, 257, 2048, 2049)] == [1, 4, 4, 16]  # the mean where no depth is known
    assert waves(1, 16, 16, 4, 7) == 4 and waves(1, 8, 8) == 1
    # A bare job list (neither known): by its workgroups.
    assert [waves(n, 0, 0) for n in (1, 4, 5, 128, 129)] == [16, 16, 4, 4, 1]
    assert waves(0, 0, 0) == -1 and waves(1, 2, 2, d=72) == -2
