"""GPU parity of the workgroup split's merge (every chunk rotation, idle waves,
whole segments, columns of several queries) and of the kernels' divisions by
block size, group and heads that are no powers of two.  Bounds are the
attention tolerances (``paged_cases.tolerances``)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import light_vllm_amd as lv
from paged_cases import DTYPES, dense_oracle_attention, make_step, tolerances

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)


@pytest.mark.parametrize("split", (True, False))
@pytest.mark.parametrize("hq,hkv,d,bs,dtype", [
    (7, 1, 128, 16, "bf16"), (6, 2, 32, 1, "fp16"), (9, 3, 48, 3, "bf16"), (5, 5, 64, 12, "fp32"), (10, 2, 80, 100, "fp16"),
    (3, 1, 96, 7, "fp32"), (4, 2, 112, 16, "fp16"), (6, 3, 144, 5, "bf16"), (5, 1, 256, 24, "fp16"), (2, 1, 256, 16, "fp32"),
])
def test_split_workgroups_match_the_dense_oracle(split, hq, hkv, d, bs, dtype) -> None:
    most = 118 if d <= 128 else 61  # (one 16-token tile a wave at four waves a workgroup)
    computed = [min(n, most) for n in (0, 1, 31, 32, 33, 63, 64, 97, 118, 77)]
    layouts = [(-1,)] * 8 + [(-1, 0), (-1, 0, 0)]  # (one column tile: at most 16 / group queries)
    if 3 * (hq // hkv) > 16:
        layouts[9] = (-1, 0)
    step = make_step(hq=hq, hkv=hkv, d=d, bs=bs, dtype=DTYPES[dtype], computed=computed, layouts=layouts, seed=d + bs)
    ctx = lv.HipPagedAttentionBackend(decode_workgroups=split).create(step.cache, step.metadata)
    out = ctx.forward(step.layer_ids[0], step.query, step.key, step.value, scale=step.scale)
    work = ctx.work_of(step.cache.layer_spec(step.layer_ids[0]))
    assert (work.group_waves > 1) == split
    err = np.abs(out.float().cpu().numpy() - dense_oracle_attention(step, step.layer_ids[0]))
    max_tol, mean_tol = tolerances(DTYPES[dtype])
    assert err.max() <= max_tol and err.mean() <= mean_tol
