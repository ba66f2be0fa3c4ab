"""The training forms of ``Linear``, ``MLP`` and ``PolarAttention`` under ``torch.compile``: one graph (``fullgraph=True``),
in which they stay the eager form; its outputs and gradients agree with those of the eager form run by itself (a call that
a dispatch mode listens to takes it too)."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from helpers import rel_err

pytestmark = pytest.mark.gpu


class Listen(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _make(kind, dev, params):
    from atma_amd.layers.global_attention import MLP, Linear, PolarAttention
    torch.manual_seed(2)
    m = {"linear": lambda: Linear(256, 512), "mlp": lambda: MLP(256),
         "attention": lambda: PolarAttention(256, head_dim=64, num_kv_heads=2)}[kind]()
    with torch.no_grad():
        for n, p in m.named_parameters():
            if p.dim() > 1:
                p.normal_(std=0.3 if "canon" in n else 0.05)
    return m.to(dev, params)


@pytest.mark.parametrize("params", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["linear", "mlp", "attention"])
def test_one_graph(dev, kind, params):
    m = _make(kind, dev, params)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 70, 256, generator=g).to(dev).bfloat16().requires_grad_(True)
    with Listen():
        y = m(x)
    go = torch.randn(y.shape, generator=g).to(dev).bfloat16()
    wrt = [x, *m.parameters()]
    want = [y, *torch.autograd.grad(y, wrt, go)]
    torch._dynamo.reset()
    z = torch.compile(m, backend="aot_eager", fullgraph=True)(x)
    got = [z, *torch.autograd.grad(z, wrt, go)]
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype
        assert rel_err(a, b) <= 4 * 2 ** -8, i   # the same products; the compiler may round a sum elsewhere
