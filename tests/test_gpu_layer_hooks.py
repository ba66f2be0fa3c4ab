"""The serving layer calls the modules that a program has changed: a hook, a patched ``forward`` or an adapter around a
projection takes part in every 16-bit inference route, and the routes' results follow it."""

import pytest
import torch
from torch import nn

from helpers import rel_err

pytestmark = pytest.mark.gpu
MODULES = ["w_gamma", "w_beta", "proj", "mu_proj", "mem.proj", "mem"]


def _layer(dev):
    from atma_amd.layers.global_attention import PolarAttention
    torch.manual_seed(7)
    layer = PolarAttention(256, head_dim=64, num_kv_heads=2)
    with torch.no_grad():
        for n, p in layer.named_parameters():
            if p.dim() > 1:
                p.normal_(std=0.3 if "canon" in n else 0.05)
    return layer.to(dev, torch.bfloat16)


def _call(layer, route, dev):
    from atma_amd.layers.global_attention import GlobalLayerCache
    g = torch.Generator().manual_seed(8)
    T, page = 40, 16
    x = torch.randn(1, T, 256, generator=g).to(dev).bfloat16()
    if route == "forward":
        return layer(x)
    cache = GlobalLayerCache.allocate(layer, 6, page, 3, dev, torch.bfloat16)
    for t in (cache.k_cache, cache.v_cache, cache.conv_q, cache.conv_k, cache.conv_v, cache.mem_table):
        t.copy_(0.3 * torch.randn(t.shape, generator=g))
    rows, pages = torch.tensor([2], device=dev), torch.tensor([[4, 0, 5, 1, 2]], dtype=torch.int32, device=dev)
    n = 24 if route == "continue" else 0
    at = torch.arange(n, n + T)
    slots = (pages[0].cpu()[at // page] * page + at % page).int().to(dev)
    if route == "continue":
        return layer.prefill_continue(x, cache, rows, slots, pages, [n])
    return layer.prefill(x, cache, rows, slots)


def _get(layer, name):
    return layer.get_submodule("mem." + name if name.startswith("w_") else name)


class Adapter(nn.Module):
    """The base layer plus its own term, the base weights exposed."""

    def __init__(self, base):
        super().__init__()
        self.base = base
        self.weight, self.bias = base.weight, base.bias

    def forward(self, x):
        return self.base(x) * 3


@pytest.mark.parametrize("route", ["continue", "prefill", "forward"])
@pytest.mark.parametrize("name", MODULES)
@torch.no_grad()
def test_hook_takes_part(dev, route, name):
    """A hook that changes the output, a patched ``forward`` and an adapter give one result, and not the unchanged layer's."""
    base = _call(_layer(dev), route, dev)
    triple = lambda y: (3 * y[0], y[1]) if isinstance(y, tuple) else 3 * y  # noqa: E731
    hooked, patched = _layer(dev), _layer(dev)
    _get(hooked, name).register_forward_hook(lambda m, i, y: triple(y))
    m = _get(patched, name)
    inner = m.forward
    m.forward = lambda *a, **k: triple(inner(*a, **k))
    outs = [_call(hooked, route, dev), _call(patched, route, dev)]
    if name != "mem":
        adapted = _layer(dev)
        parent, _, leaf = ("mem." + name if name.startswith("w_") else name).rpartition(".")
        setattr(adapted.get_submodule(parent), leaf, Adapter(_get(adapted, name)))
        outs.append(_call(adapted, route, dev))
    for y in outs:
        assert torch.equal(y, outs[0])
    assert rel_err(outs[0], base) > 0.05   # far above the routes' roundings (2^-8 each)


@pytest.mark.parametrize("route", ["continue", "prefill", "forward"])
@torch.no_grad()
def test_hook_that_only_looks_changes_little(dev, route):
    layer, seen = _layer(dev), []
    base = _call(layer, route, dev)
    for name in MODULES:
        _get(layer, name).register_forward_hook(lambda m, i, y, name=name: seen.append(name))
    y = _call(layer, route, dev)
    assert sorted(set(seen)) == sorted(MODULES)
    assert rel_err(y, base) <= 6 * 2 ** -8   # a few 16-bit roundings in other places
