"""Calls that skip the dispatcher: the same results as the registered op, version counters advanced alike, and the
dispatcher kept wherever something listens to it."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


def _args(dev):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(5, 64, generator=g).bfloat16().to(dev)
    table = torch.randn(7, 64, 3, generator=g).bfloat16().to(dev)
    w = torch.randn(64, 4, generator=g).bfloat16().to(dev)
    return x, w, torch.tensor([6, 0, 2, 5, 1], device=dev), table


def test_direct_equals_dispatched(dev):
    from atma_amd import _ops
    x, w, slots, table = _args(dev)
    t1, t2 = table.clone(), table.clone()
    with torch.no_grad():
        v1, v2 = t1._version, t2._version
        a = _ops.run.causal_conv1d_decode_step(x, w, slots, t1, True)
        b = torch.ops.atma_hip.causal_conv1d_decode_step(x, w, slots, t2, True)
    assert torch.equal(a, b) and torch.equal(t1, t2) and not torch.equal(t1, table)
    assert t1._version - v1 == t2._version - v2 > 0
    with torch.inference_mode():   # inference tensors have no version counter
        _ops.run.causal_conv1d_decode_step(x, w, slots, table.clone(), True)
        _ops.run.causal_conv1d_decode_step(x, w, slots, t1, True)


def test_who_listens_gets_the_op(dev):
    from atma_amd import _ops
    x, w, slots, table = _args(dev)
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with torch.no_grad(), Log():
        _ops.run.causal_conv1d_decode_step(x, w, slots, table, True)
    assert any("causal_conv1d_decode_step" in s for s in seen)
    assert not _ops._undispatched((x.clone().requires_grad_(),)) and _ops._undispatched((x, [x, w], 3, None))
    with torch.no_grad():
        assert _ops._undispatched((x.clone().requires_grad_(),))

    class Sub(torch.Tensor):
        pass

    assert not _ops._undispatched((x.as_subclass(Sub),)) and not _ops._undispatched(([x.as_subclass(Sub)],))
    with pytest.raises(RuntimeError, match="GPU only"):
        _ops.run.causal_conv1d_decode_step(x.cpu(), w, slots, table, True)
