"""GPU parity of the split-K merge's shapes: a few partials per job (one wave
per column set), some (four waves share a job's partials) and many (sixteen
do), with columns that leave part of a wave or workgroup idle, at row widths
from four to sixty-four lanes per column.  Bounds are the attention
tolerances (``paged_cases.tolerances``)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import light_vllm_amd as lv
from light_vllm_amd import native
from light_vllm_amd.paged_cache import dtype_code
from paged_cases import DTYPES, dense_oracle_attention, make_step, tolerances

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)

# (computed tokens of each sequence, fewest and most partials per merge job on average)
DEPTHS = {
    "few": ([700, 901, 650, 777, 1100] * 40, 1, 8),
    "some": ([900, 33, 700, 1203] * 7, 8, 32),
    "many": ([8111], 32, 256),
    "many_uneven": ([5003, 40], 32, 256),
}


@pytest.mark.parametrize("hq,hkv,d,dtype", [(7, 1, 128, "bf16"), (10, 2, 80, "fp16"), (3, 1, 32, "bf16"),
                                            (5, 1, 256, "fp32"), (14, 2, 64, "fp32"), (3, 3, 192, "fp16")])
@pytest.mark.parametrize("depth", DEPTHS)
def test_merge_shapes_match_the_dense_oracle(depth, hq, hkv, d, dtype) -> None:
    computed, lo, hi = DEPTHS[depth]
    step = make_step(hq=hq, hkv=hkv, d=d, bs=16, dtype=DTYPES[dtype], computed=computed, layouts=[(-1,)] * len(computed),
                     seed=len(depth) + d)
    ctx = lv.HipPagedAttentionBackend(decode_workgroups=False).create(step.cache, step.metadata)
    out = ctx.forward(step.layer_ids[0], step.query, step.key, step.value, scale=step.scale)
    work = ctx.work_of(step.cache.layer_spec(step.layer_ids[0]))
    if hkv == 1 and d <= 128:  # (other shapes have other tiles and resident waves)
        assert lo < work.num_partial_slots / work.num_jobs <= hi
    err = np.abs(out.float().cpu().numpy() - dense_oracle_attention(step, step.layer_ids[0]))
    max_tol, mean_tol = tolerances(DTYPES[dtype])
    assert err.max() <= max_tol and err.mean() <= mean_tol


# One deep job among shallow ones, by the depth that the plan knows: within a
# round trip of four and of sixteen waves, and beyond one of four (64 jobs, too
# many columns for sixteen).
@pytest.mark.parametrize("computed, hq, hkv, d, dtype, shape, rounds", (
    ([2500] + [200] * 31, 7, 1, 128, "bf16", 16, 1), ([1500] + [40] * 20, 7, 1, 128, "bf16", 4, 1),
    ([9000] + [300] * 63, 28, 4, 128, "bf16", 4, 2), ([9000] + [120] * 300, 4, 1, 256, "fp16", 4, 2),
    ([5000] + [100] * 40, 5, 1, 80, "fp16", 16, 1)))
def test_one_deep_job_among_shallow_ones(computed, hq, hkv, d, dtype, shape, rounds) -> None:
    step = make_step(hq=hq, hkv=hkv, d=d, bs=16, dtype=DTYPES[dtype], computed=computed,
                     layouts=[(-1,)] * len(computed), seed=d)
    ctx = lv.HipPagedAttentionBackend(decode_workgroups=False).create(step.cache, step.metadata)
    out = ctx.forward(step.layer_ids[0], step.query, step.key, step.value, scale=step.scale)
    work = ctx.work_of(step.cache.layer_spec(step.layer_ids[0]))
    assert work.merge_depth == int(work.jobs.cpu().numpy()[:, 3].max())
    waves = native.load().lvamd_paged_merge_waves(dtype_code(DTYPES[dtype]), d, work.num_jobs, work.num_partial_slots,
                                                  work.merge_depth, hkv, work.merge_columns)
    assert waves == shape and -(-work.merge_depth // (16 * waves)) >= rounds
    err = np.abs(out.float().cpu().numpy() - dense_oracle_attention(step, step.layer_ids[0]))
    max_tol, mean_tol = tolerances(DTYPES[dtype])
    assert err.max() <= max_tol and err.mean() <= mean_tol
