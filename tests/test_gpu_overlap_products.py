"""The overlapped schedule makes no library product on the main stream while the memory branch makes its own on the other."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("route", ["forward", "continue"])
@torch.no_grad()
def test_products_after_the_join(dev, monkeypatch, dtype, route):
    from atma_amd.layers.global_attention import GlobalLayerCache, PolarAttention
    layer = PolarAttention(256, head_dim=64, num_kv_heads=2, overlap=True).to(dev, dtype)
    x = torch.randn(1, 40, 256, device=dev, dtype=dtype)
    cache = GlobalLayerCache.allocate(layer, 4, 16, 3, dev, dtype)
    at = torch.arange(40).int().to(dev)
    pages = torch.arange(4, dtype=torch.int32, device=dev)[None]
    log, wait, linear = [], torch.cuda.Stream.wait_stream, torch.nn.functional.linear
    monkeypatch.setattr(torch.cuda.Stream, "wait_stream", lambda s, other: (log.append("wait"), wait(s, other))[1])
    main = torch.cuda.current_stream(dev)
    monkeypatch.setattr(torch.nn.functional, "linear", lambda *a: (
        log.append("main" if torch.cuda.current_stream(dev) == main else "side"), linear(*a))[1])
    for name in ("proj", "mu_proj"):   # hooked: the 16-bit layer calls them too
        layer.get_submodule(name).register_forward_hook(lambda *a: None)
    if route == "forward":
        layer(x)
    else:
        layer.prefill_continue(x, cache, torch.tensor([1], device=dev), at, pages, [0])
    assert log.count("wait") == 2, log
    first, last = log.index("wait"), len(log) - 1 - log[::-1].index("wait")
    assert "side" in log[first:last] and "main" not in log[first:last] and log[last:].count("main") >= 2, log
