"""The prefill routes write conv tails, KV pages and states in place: what asks for a tensor's version sees it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_prefill_advances_versions(dev, dtype):
    from atma_amd.layers.global_attention import GlobalLayerCache, PolarAttention
    layer = PolarAttention(256, head_dim=64, num_kv_heads=2).to(dev, dtype)
    x = torch.randn(1, 20, 256, device=dev, dtype=dtype)
    cache = GlobalLayerCache.allocate(layer, 4, 16, 3, dev, dtype)
    tables = [cache.k_cache, cache.v_cache, cache.conv_q, cache.conv_k, cache.conv_v, cache.mem_table]
    rows, pages = torch.tensor([1], device=dev), torch.tensor([[2, 0, 1]], dtype=torch.int32, device=dev)
    slots = (pages[0].cpu()[torch.arange(40) // 16] * 16 + torch.arange(40) % 16).int().to(dev)
    for call in (lambda: layer.prefill(x, cache, rows, slots[:20]),
                 lambda: layer.prefill_continue(x, cache, rows, slots[20:], pages, [20])):
        before = [t._version for t in tables]
        with torch.no_grad():
            call()
        assert all(t._version > b for t, b in zip(tables, before))
    w = torch.ones_like(cache.conv_q, requires_grad=True)
    y = (w * cache.conv_q).sum()   # saves the table for w's gradient
    with torch.no_grad():
        layer.prefill(x, cache, rows, slots[:20])
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()
    with torch.inference_mode():   # inference tensors have no version
        layer.prefill(x, GlobalLayerCache.allocate(layer, 4, 16, 3, dev, dtype), rows, slots[:20])
