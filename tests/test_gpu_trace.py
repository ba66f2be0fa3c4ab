"""The layer's inference routes under ``torch.jit.trace``: what is recorded answers inputs and parameters other than those
it was traced with.  The replay repeats what the eager call does where it is recorded (torch and registered ops, the same
kernels), so it is compared with that bit for bit, and with the fused eager call to the roundings that differ: a few
16-bit ones of values of the output's size (2^-8 each), none in fp32 beyond the sums' order."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from helpers import polar_params, rel_err

pytestmark = pytest.mark.gpu
BOUND = {torch.float32: 1e-4, torch.bfloat16: 6 * 2 ** -8}


class Listen(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _layer(dev, dtype):
    from atma_amd.layers.global_attention import PolarAttention
    torch.manual_seed(5)
    layer = PolarAttention(256, head_dim=64, num_kv_heads=2)
    with torch.no_grad():
        for n, p in layer.named_parameters():
            if p.dim() > 1:
                p.normal_(std=0.3 if "canon" in n else 0.05)
    return layer.to(dev, dtype).requires_grad_(False)   # (a trace takes no constant that requires grad)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_traced_forward(dev, dtype):
    layer = _layer(dev, dtype)
    x, y = (torch.randn(2, 70, 256, generator=torch.Generator().manual_seed(s)).to(dev, dtype) for s in (1, 2))
    traced = torch.jit.trace(lambda t: layer(t), (x,), check_trace=False)
    layer.v_null.mul_(-2)   # read at the replay, not kept from the trace
    with Listen():
        want = layer(y)
    assert torch.equal(traced(y), want)
    assert rel_err(want, layer(y)) <= BOUND[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_traced_continue(dev, dtype):
    from atma_amd.layers.global_attention import GlobalLayerCache
    layer = _layer(dev, dtype)
    g = torch.Generator().manual_seed(3)
    T, n, page = 20, 40, 16
    cache = GlobalLayerCache.allocate(layer, 6, page, 3, dev, dtype)
    for t in (cache.k_cache, cache.v_cache, cache.conv_q, cache.conv_k, cache.conv_v, cache.mem_table):
        t.copy_(0.3 * torch.randn(t.shape, generator=g))
    rows, pages = torch.tensor([2], device=dev), torch.tensor([[4, 0, 5, 1]], dtype=torch.int32, device=dev)
    at = torch.arange(n, n + T)
    slots = (pages[0].cpu()[at // page] * page + at % page).int().to(dev)
    names = ("k_cache", "v_cache", "conv_q", "conv_k", "conv_v", "mem_table")
    kept = [getattr(cache, m) for m in names]

    def call(t, *tables):   # (inputs of the trace: it drops writes to what it holds as constants)
        return layer.prefill_continue(t, GlobalLayerCache(**dict(zip(names, tables))), rows, slots, pages, [n])

    def run(fn, t):
        tables = [a.clone() for a in kept]
        return [fn(t, *tables)] + tables

    x, y = (torch.randn(1, T, 256, generator=g).to(dev, dtype) for _ in range(2))
    traced = torch.jit.trace(call, (x, *(a.clone() for a in kept)), check_trace=False)
    with Listen():
        want = run(call, y)
    got, fused = run(traced, y), run(call, y)
    for a, b, c in zip(got, want, fused):
        assert torch.equal(a, b)
        assert rel_err(b, c) <= BOUND[dtype]


@torch.no_grad()
def test_traced_polar_reads_its_parameters(dev):
    """16-bit parameters, widened by a launch of their own outside a trace."""
    from atma_amd.kernel import polar_attention_fwd
    H, Hkv, T, d = 4, 2, 33, 64
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(1, h, T, d, generator=g).to(dev).bfloat16() for h in (H, Hkv, Hkv))
    n = torch.arange(1, T + 1, dtype=torch.float32, device=dev)
    p = [list(polar_params(H, d, seed=s, dtype=torch.bfloat16, device=dev).values()) for s in (0, 1)]

    def call(*ps):
        return polar_attention_fwd(q, k, v, n, v_null=ps[0], null_base=ps[1], null_slope_raw=ps[2], len_gain_raw=ps[3],
                                   mag_beta_raw=ps[4])

    traced = torch.jit.trace(call, tuple(p[0]), check_trace=False)
    for got, want in zip(traced(*p[1]), call(*p[1])):
        assert torch.equal(got, want)


@torch.no_grad()
def test_traced_mlp(dev):
    """Rows enough for the projection and its activation as one kernel (4,096) outside a trace."""
    from atma_amd.layers.global_attention import MLP
    torch.manual_seed(6)
    mlp = MLP(128).to(dev, torch.bfloat16).requires_grad_(False)
    x, y = (torch.randn(4096, 128, generator=torch.Generator().manual_seed(s)).to(dev).bfloat16() for s in (1, 2))
    traced = torch.jit.trace(lambda t: mlp(t), (x,), check_trace=False)
    got = traced(y)   # (before the eager call, whose freed buffers would hold the answer)
    with Listen():
        want = mlp(y)
    assert torch.equal(got, want)
    assert rel_err(want, mlp(y)) <= BOUND[torch.bfloat16]
