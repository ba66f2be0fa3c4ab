"""A call that skips the dispatcher is not made where the JIT tracer records: the traced graph holds the op's node and
answers other inputs than those it was traced with, in-place writes included."""

import pytest
import torch

from atma_amd import _ops


@pytest.fixture(scope="module")
def probe():
    """An op whose writes torch does not see, as a native launch's are not."""
    if not hasattr(_ops.run, "trace_probe"):
        @_ops._op("trace_probe", mutates_args=("table",))
        def trace_probe(x: torch.Tensor, table: torch.Tensor) -> torch.Tensor:
            out = torch.empty_like(x)
            out.numpy()[:] = 2 * x.numpy()
            table.numpy()[:] += 1
            return out

        @trace_probe.register_fake
        def _(x, table):
            return torch.empty_like(x)
    return _ops.run.trace_probe


@pytest.mark.parametrize("grad_mode", [False, True])
def test_traced_op_replays(probe, grad_mode):
    with torch.set_grad_enabled(grad_mode):
        traced = torch.jit.trace(lambda x, t: probe(x, t) + 0, (torch.ones(3), torch.zeros(2)), check_trace=False)
    assert "atma_hip::trace_probe" in str(traced.graph)
    table = torch.zeros(2)
    for i in range(2):
        assert torch.equal(traced(torch.tensor([1., 2., 3.]) + i, table), 2 * (torch.tensor([1., 2., 3.]) + i))
    assert torch.equal(table, torch.full((2,), 2.))


def test_watched():
    seen = []

    def f(x):
        seen.append(_ops.watched())
        return x + 1

    assert not _ops.watched()
    torch.jit.trace(f, (torch.ones(2),), check_trace=False)
    torch.func.vmap(f)(torch.ones(2, 2))
    torch.func.jvp(f, (torch.ones(2),), (torch.ones(2),))
    with torch.device("cpu"):   # a function mode records nothing
        f(torch.ones(2))
    assert seen == [True, True, True, False] and not _ops.watched()
