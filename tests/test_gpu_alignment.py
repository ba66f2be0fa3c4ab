"""Parameters, gradients and caches that are views at an odd offset of a larger buffer: what the kernels' 16-byte accesses
cannot take is copied or left to the eager form, and the results are those of the same values at aligned addresses (bit
for bit where the same kernels run, else to a few 16-bit roundings, 2^-8 of the largest value each)."""

import pytest
import torch

from helpers import rel_err

pytestmark = pytest.mark.gpu
FEW = 6 * 2 ** -8


def _odd(t):
    """The values of t one element into a buffer."""
    flat = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 and out.is_contiguous()
    return out


def _module(kind, dev, dtype):
    from atma_amd.layers.global_attention import MLP, Linear, PolarAttention
    torch.manual_seed(11)
    m = {"linear": lambda: Linear(256, 512), "mlp": lambda: MLP(256),
         "attention": lambda: PolarAttention(256, head_dim=64, num_kv_heads=2)}[kind]()
    with torch.no_grad():
        for n, p in m.named_parameters():
            if p.dim() > 1:
                p.normal_(std=0.3 if "canon" in n else 0.05)
    return m.to(dev, dtype)


def _misalign(m):
    for name, p in m.named_parameters():
        if name.endswith(("weight", "bias")):
            p.data = _odd(p.data)
    return m


@pytest.mark.parametrize("params", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["linear", "mlp", "attention"])
def test_parameters_in_training(dev, kind, params):
    g = torch.Generator().manual_seed(12)
    x = torch.randn(2, 70, 256, generator=g).to(dev).bfloat16().requires_grad_(True)
    res = []
    for m in (_module(kind, dev, params), _misalign(_module(kind, dev, params))):
        y = m(x)
        if not res:
            go = torch.randn(y.shape, generator=g).to(dev).bfloat16()
        res.append([y, *torch.autograd.grad(y, [x, *m.parameters()], go)])
    for i, (a, b) in enumerate(zip(*res)):
        assert rel_err(b, a) <= 2 * FEW, i   # forward and backward


@pytest.mark.parametrize("rows", [1, 70])
def test_gradients(dev, rows):
    """Output gradients at odd offsets, and rows of one with an odd stride."""
    from atma_amd.kernel.canon import canon_conv
    from atma_amd.kernel.train_glue import (gate_train, head_norm_train, linear_train, out_train, project_train,
                                            squared_relu_gate_train)
    from atma_amd.layers.global_attention import Linear
    H, d = 4, 64
    g = torch.Generator().manual_seed(rows)

    def r(*shape):
        return torch.randn(*shape, generator=g).to(dev).bfloat16().requires_grad_(True)

    x = r(rows, 256)
    lin = [Linear(256, n).to(dev) for n in (2 * H * d, 128, 64)]
    out = [Linear(128, 256).to(dev) for _ in range(2)]
    c = r(1, H, rows, d)
    calls = [
        (lambda: linear_train(x, lin[1].weight, lin[1].bias), [x, lin[1].weight, lin[1].bias]),
        (lambda: project_train(x, lin, d), [x, *(p for m in lin for p in m.parameters())]),
        (lambda: out_train(x, out), [x, *(p for m in out for p in m.parameters())]),
        (lambda: squared_relu_gate_train(x), [x]),
    ]
    q, k, gate, rr, mg = r(rows, H, d), r(rows, 2, d), r(rows, H, d), r(rows, H, d), r(rows, H * d)
    calls.append((lambda: head_norm_train(q, k, 1e-6), [q, k]))
    calls.append((lambda: gate_train(c.transpose(1, 2), gate, rr, mg, 1e-6), [c, gate, rr, mg]))
    cs, ws = [r(1, rows, n * d) for n in (H, 2, 2)], [r(n * d, 1, 4) for n in (H, 2, 2)]
    calls.append((lambda: canon_conv(*cs, *ws), [*cs, *ws]))
    for i, (fn, wrt) in enumerate(calls):
        ys = fn()
        ys = ys if isinstance(ys, tuple) else (ys,)
        gs = [torch.randn(y.shape, generator=g).to(dev).bfloat16() for y in ys]
        want = torch.autograd.grad(ys, wrt, gs)

        def wide(t):   # a slice of wider rows: an odd stride between rows, aligned only where it starts
            buf = torch.zeros(*t.shape[:-1], t.shape[-1] + 3, device=dev, dtype=t.dtype)
            buf[..., :t.shape[-1]] = t
            return buf[..., :t.shape[-1]]

        for form in (_odd, wide):
            got = torch.autograd.grad(fn(), wrt, [form(t) for t in gs])
            for a, b in zip(got, want):
                assert torch.equal(a, b), (i, form.__name__)


@pytest.mark.parametrize("what", ["canon", "caches", "parameters"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@torch.no_grad()
def test_serving_routes(dev, dtype, what):
    from atma_amd.layers.global_attention import GlobalLayerCache
    g = torch.Generator().manual_seed(13)
    T, page = 40, 16
    x = torch.randn(1, T, 256, generator=g).to(dev, dtype)
    fill = None
    res = []
    for odd in (False, True):
        layer = _module("attention", dev, dtype)
        if odd and what != "caches":
            for name, p in layer.named_parameters():
                if "canon" in name or (what == "parameters" and name.endswith(("weight", "bias"))):
                    p.data = _odd(p.data)
        cache = GlobalLayerCache.allocate(layer, 8, page, 3, dev, dtype)
        tables = [cache.k_cache, cache.v_cache, cache.conv_q, cache.conv_k, cache.conv_v, cache.mem_table]
        fill = fill or [0.3 * torch.randn(t.shape, generator=g) for t in tables]
        for t, f in zip(tables, fill):
            t.copy_(f)
        if odd and what == "caches":
            cache.k_cache, cache.v_cache = _odd(cache.k_cache), _odd(cache.v_cache)
        rows, pages = torch.tensor([2], device=dev), torch.tensor([[4, 0, 5, 1, 2, 7]], dtype=torch.int32, device=dev)
        outs = [layer(x)]
        for n in (0, T):
            at = torch.arange(n, n + T)
            slots = (pages[0].cpu()[at // page] * page + at % page).int().to(dev)
            outs.append(layer.prefill(x, cache, rows, slots) if n == 0 else
                        layer.prefill_continue(x, cache, rows, slots, pages, [n]))
        res.append(outs + [cache.k_cache, cache.v_cache, cache.conv_q, cache.conv_k, cache.conv_v, cache.mem_table])
    for i, (a, b) in enumerate(zip(*res)):
        assert rel_err(b, a) <= (1e-5 if dtype == torch.float32 else FEW), i


@torch.no_grad()
def test_deferred_sum(dev):
    from atma_amd.kernel.decode_fusions import PartialSums
    g = torch.Generator().manual_seed(14)
    M, D, k = 5, 256, 4
    base, mu_x, mu_w, bias = (torch.randn(*s, generator=g).to(dev).bfloat16() for s in ((M, D), (M, k), (D, k), (D,)))
    want = PartialSums(None, [bias], mu_x=mu_x, mu_w=mu_w, base=base).materialize()
    assert rel_err(want, base.double() + bias.double() + mu_x.double() @ mu_w.double().t()) <= 2 ** -8
    one = torch.empty_strided((1, k), (1, 1), device=dev, dtype=base.dtype).copy_(mu_x[:1])
    for ps, rows in ((PartialSums(None, [bias], mu_x=mu_x, mu_w=_odd(mu_w), base=base), M),
                     (PartialSums(None, [_odd(bias)], mu_x=mu_x, mu_w=mu_w, base=base), M),
                     (PartialSums(None, [bias], mu_x=mu_x, mu_w=mu_w, base=_odd(base)), M),
                     (PartialSums(None, [bias], mu_x=one, mu_w=mu_w, base=base[:1]), 1)):
        assert rel_err(ps.materialize(), want[:rows]) <= 2 ** -7   # one rounding each
