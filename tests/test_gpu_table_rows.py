"""Negative table rows of a continued chunk count from the end, in the conv tails as in the memory's states."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [2, 20])
@torch.no_grad()
def test_continue_counts_rows_from_the_end(dev, dtype, T):
    from atma_amd.layers.global_attention import GlobalLayerCache, PolarAttention
    torch.manual_seed(41)
    layer = PolarAttention(256, head_dim=64, num_kv_heads=2).to(dev, dtype)
    n, page, R = 24, 16, 5
    g = torch.Generator().manual_seed(42)
    x = torch.randn(2, T, 256, generator=g).to(dev, dtype)
    pages = torch.tensor([[4, 0, 5], [1, 6, 2]], dtype=torch.int32, device=dev)
    at = torch.arange(n, n + T)
    slots = torch.cat([p[at // page] * page + at % page for p in pages.cpu()]).int().to(dev)
    cache = GlobalLayerCache.allocate(layer, 7, page, R, dev, dtype)
    names = ("k_cache", "v_cache", "conv_q", "conv_k", "conv_v", "mem_table")
    kept = [0.3 * torch.randn(getattr(cache, m).shape, generator=g) for m in names]
    res = []
    for rows in ([R - 1, 1], [-1, 1 - R]):
        for m, t in zip(names, kept):
            getattr(cache, m).copy_(t)
        y = layer.prefill_continue(x, cache, torch.tensor(rows, device=dev), slots, pages, [n, n])
        res.append([y] + [getattr(cache, m).clone() for m in names])
    for a, b in zip(*res):
        assert torch.equal(a, b)
    for m, t, now in zip(names[2:], kept[2:], res[1][3:]):   # the other rows stay
        assert torch.equal(now[[0, 2, 3]].cpu(), t[[0, 2, 3]].to(now.dtype)) and not torch.equal(now[4].cpu(), t[4].to(now.dtype))
