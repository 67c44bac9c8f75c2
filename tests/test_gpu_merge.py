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


@pytest.mark.parametrize("jobs, waves", ((1, 16), (10, 16), (11, 4), (341, 4), (342, 1)))
@pytest.mark.parametrize("d, dtype", ((128, "bf16"), (48, "fp16"), (112, "fp32")))
def test_bare_job_list(jobs, waves, d, dtype) -> None:
    """The separate merge entry on made-up partials: its first job deeper than
    a round trip of every shape, one partial empty.  A result is the weighted
    mean of rows already in the pool's type, so it may differ by its own
    rounding and by fp32 sums of 300 terms."""
    hkv, group = 3, 2
    assert native.load().lvamd_paged_merge_waves(dtype_code(DTYPES[dtype]), d, jobs, 0, 0, hkv, group) == waves
    depth = [300] + [1 + i % 5 for i in range(jobs - 1)]
    rng = np.random.default_rng(jobs)
    start = np.cumsum([0] + depth)
    records = torch.tensor([[i, 0, start[i], n, i, 1, 0, 0] for i, n in enumerate(depth)], dtype=torch.int32).cuda()
    acc = torch.from_numpy(rng.standard_normal((start[-1], hkv, 16, d), dtype=np.float32)).to(DTYPES[dtype]).cuda()
    pairs = np.stack((rng.uniform(-6, 6, (start[-1], hkv, 16)), rng.uniform(1, 9, (start[-1], hkv, 16))), -1)
    pairs[7] = (-np.inf, 0.0)
    ml = torch.from_numpy(pairs.astype(np.float32)).cuda()
    out = torch.empty((jobs, hkv * group, d), dtype=DTYPES[dtype], device="cuda:0")
    native.check(native.load().lvamd_paged_attention_merge(
        acc.data_ptr(), ml.data_ptr(), out.data_ptr(), out.stride(0), out.stride(1), records.data_ptr(), jobs, hkv, group,
        d, 1, group, dtype_code(DTYPES[dtype]), torch.cuda.current_stream().cuda_stream), "lvamd_paged_attention_merge")
    rows, stats = acc.double().cpu().numpy()[:, :, :group], ml.double().cpu().numpy()[:, :, :group]
    unit = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 2.0 ** -24}[dtype]  # 2 ** -p: p significant bits, to nearest
    for i in range(jobs):
        m = stats[start[i]:start[i + 1]]
        weight = np.exp2(m[..., 0] - m[..., 0].max(0)) * m[..., 1]
        part = rows[start[i]:start[i + 1]] * weight[..., None]
        want = (part.sum(0) / weight.sum(0)[..., None]).reshape(hkv * group, d)
        size = (np.abs(part).sum(0) / weight.sum(0)[..., None]).reshape(hkv * group, d)
        bound = unit * np.abs(want) + 400 * 2.0 ** -24 * size + 2.0 ** -24  # (last: fp16 below its normal range)
        excess = (np.abs(out[i].double().cpu().numpy() - want) - bound).max()
        assert excess <= 0, i
