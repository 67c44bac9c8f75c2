"""GPU test: forward(rotary=) by its native call equals the general path bit
for bit (outputs and pool rows), for own and projection-view Q/K/V, strided
cosine rows, several layers and streams; what the native call does not take
(unaligned rows, a list of tensors) still runs, and broken rules still raise."""

from __future__ import annotations

import pytest
import torch

import light_vllm_amd as lv
from paged_cases import DTYPES, make_step

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)


def _rows(tokens: int, d: int, dtype, strided: bool):
    gen = torch.Generator(device="cuda:0").manual_seed(tokens)
    rows = torch.randn((tokens, 2 * d), generator=gen, device="cuda:0").to(dtype)
    return (rows[:, :d], rows[:, d:]) if strided else (rows[:, :d].contiguous(), rows[:, d:].contiguous())


def _count_general(ctx) -> list[str]:
    """The layers that take the general path from here on."""
    taken, forward = [], ctx._forward_general

    def counted(layer_id, *args, **kw):
        taken.append(layer_id)
        return forward(layer_id, *args, **kw)

    ctx._forward_general = counted
    return taken


def _run(case, general: bool, views: bool, strided: bool, streams: bool = False):
    step = make_step(**case)
    pools = [t for lid in step.layer_ids for t in (step.cache.layer(lid).keys, step.cache.layer(lid).values)]
    held = torch.zeros(pools[0].shape[:2], dtype=torch.bool)  # the step's cached rows; every other row starts at 0
    for table, n in zip(step.metadata.block_tables, case["computed"]):
        for i in range(n):
            held[table[i // case["bs"]], i % case["bs"]] = True
    for t in pools:
        t[~held.cuda()] = 0
    ctx = lv.HipPagedAttentionBackend().create(step.cache, step.metadata)
    generals = _count_general(ctx)
    if general:
        ctx._statics = {}  # no native call: every layer takes the general path
    tokens, d = step.query.shape[0], case["d"]
    q, k, v = step.query, step.key, step.value
    if views:
        packed = torch.cat((q, k, v), dim=1)
        hq, hkv = case["hq"], case["hkv"]
        q, k, v = packed[:, :hq], packed[:, hq : hq + hkv], packed[:, hq + hkv :]
    rotary = _rows(tokens, d, case["dtype"], strided)
    outs = []
    for i, lid in enumerate(step.layer_ids):
        side = torch.cuda.Stream() if streams and i % 2 else torch.cuda.current_stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            outs.append(ctx.forward(lid, q, k, v, scale=step.scale, rotary=rotary))
        torch.cuda.current_stream().wait_stream(side)  # (the split-K workspace is the stream's)
    torch.cuda.synchronize()
    assert len(generals) == (len(step.layer_ids) if general else 0)
    return outs, pools


@pytest.mark.parametrize("views,strided,streams", ((False, False, False), (True, True, False), (False, True, True)))
@pytest.mark.parametrize("dtype,d,bs", (("bf16", 128, 16), ("fp16", 80, 12), ("fp32", 64, 16)))
def test_native_rotary_call_equals_the_general_path(dtype, d, bs, views, strided, streams) -> None:
    case = dict(hq=6, hkv=2, d=d, bs=bs, dtype=DTYPES[dtype], computed=[300, 17, 0],
                layouts=[(-1,), (-1, 0, 1, 0), tuple(range(-1, 40))], seed=d, num_layers=3)
    got, want = (_run(case, general, views, strided, streams and not general) for general in (False, True))
    for a, b in zip(got[0], want[0]):
        assert torch.equal(a, b)
    for a, b in zip(got[1], want[1]):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_other_rotary_arguments_take_the_general_path() -> None:
    case = dict(hq=4, hkv=2, d=64, bs=16, dtype=torch.bfloat16, computed=[40], layouts=[(-1,)], seed=3, num_layers=6)
    step = make_step(**case)
    first = step.cache.layer("layer0")
    for layer in (step.cache.layer("layer1"), step.cache.layer("layer5")):
        layer.keys.copy_(first.keys)
        layer.values.copy_(first.values)
    ctx = lv.HipPagedAttentionBackend().create(step.cache, step.metadata)
    cos, sin = _rows(1, 64, torch.bfloat16, False)
    generals = _count_general(ctx)
    call = lambda i, q, r: ctx.forward(f"layer{i}", q, step.key, step.value, scale=step.scale, rotary=r)  # noqa: E731
    first = call(0, step.query, (cos, sin))
    shifted = torch.empty(4 * 64 + 1, dtype=torch.bfloat16, device="cuda:0")[1:].view(1, 4, 64).copy_(step.query)
    assert generals == []
    assert torch.equal(call(1, step.query, [cos, sin]), first)
    assert torch.equal(call(5, shifted, (cos, sin)), first)
    assert generals == ["layer1", "layer5"]
    with pytest.raises(lv.KVCacheError, match="rotary cosines must have shape"):
        call(2, step.query, (cos[:, :32], sin))
    with pytest.raises(lv.KVCacheError, match="rotary sines dtype and device"):
        call(3, step.query, (cos, sin.float()))
    with pytest.raises(lv.KVCacheError, match="rotary cosines must have shape"):
        call(4, step.query, (None, sin))
    assert generals == ["layer1", "layer5", "layer2", "layer3", "layer4"]
