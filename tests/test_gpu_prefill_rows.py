"""GPU test: the prefill kernel's ways to address the step's K/V rows.  Row
blocks of 16 in the step's input take a scalar base up to token strides of
2**24 elements and an address per lane from there on (always at D = 128 with
block sizes other than powers of two from 16); both, and rows shared by all
tokens (stride 0), equal the same rows laid out contiguously bit for bit, in
the outputs and in the pool."""

from __future__ import annotations

import pytest
import torch

import light_vllm_amd as lv
from paged_cases import make_step

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)


def _run(d: int, bs: int, queries: int, stride: int | None, spread: bool):
    # 16 cached tokens: the chunk's first row block lies wholly in the input, its last one is cut short.
    step = make_step(hq=4, hkv=2, d=d, bs=bs, dtype=torch.bfloat16, computed=[40, 16],
                     layouts=[(-1,), tuple(range(-1, queries - 1))], seed=bs)
    key, value = step.key, step.value
    if stride == 0:
        key, value = (t[:1].expand(t.shape) for t in (key, value))
        if not spread:
            key, value = key.contiguous(), value.contiguous()
    elif spread:
        key, value = (torch.empty_strided(t.shape, (stride, d, 1), dtype=t.dtype, device=t.device).copy_(t)
                      for t in (key, value))
    layer = step.cache.layer("layer0")
    held = torch.zeros(layer.keys.shape[:2], dtype=torch.bool)  # the cached rows; every other row starts at 0
    for table, n in zip(step.metadata.block_tables, (40, 16)):
        for i in range(n):
            held[table[i // bs], i % bs] = True
    for t in (layer.keys, layer.values):
        t[~held.cuda()] = 0
    ctx = lv.HipPagedAttentionBackend().create(step.cache, step.metadata)
    out = ctx.forward("layer0", step.query, key, value, scale=step.scale)
    torch.cuda.synchronize()
    return out, layer.keys, layer.values


@pytest.mark.parametrize("d", (64, 128))
@pytest.mark.parametrize("bs", (16, 32, 12))
@pytest.mark.parametrize("queries,stride", ((40, 0), (40, 264), (24, (1 << 24) - 8), (24, 1 << 24)))
def test_row_strides_of_the_step_equal_contiguous_rows(d, bs, queries, stride) -> None:
    got, want = (_run(d, bs, queries, stride, spread) for spread in (True, False))
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
