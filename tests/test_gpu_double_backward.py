"""``create_graph`` through the training launches with some of their operands frozen: the gradients' gradients of the
others, against the same composition in float64."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _double(fn, args, live):
    """Gradients of the squared first gradients with respect to args[live]."""
    xs = [a.detach().clone().requires_grad_(i in live) for i, a in enumerate(args)]
    outs = fn(*xs)
    outs = outs if isinstance(outs, tuple) else (outs,)
    # (squared: the second derivative of a linear map by itself is zero)
    loss = sum(o.to(torch.float64 if o.dtype == torch.float64 else torch.float32).square().sum() for o in outs)
    wrt = [xs[i] for i in live]
    first = torch.autograd.grad(loss, wrt, create_graph=True)
    return torch.autograd.grad(sum(g.to(loss.dtype).square().sum() for g in first), wrt)


def _check(fn, eager, args, live, tol):
    got, ref = _double(fn, args, live), _double(eager, [a.double() for a in args], live)
    for i, a, b in zip(live, got, ref):
        assert (a.double() - b).abs().max() <= tol * b.abs().max(), i


def _conv(x, w):
    return x + F.conv1d(F.pad(x.transpose(1, 2), (w.shape[-1] - 1, 0)), w, groups=x.shape[2]).transpose(1, 2)


@pytest.mark.parametrize("live", [(0, 1, 2), (3, 4, 5), (0, 4), (2,), (0, 1, 2, 3, 4, 5)])
def test_canon_conv(dev, live):
    from atma_amd.kernel.canon import canon_conv
    g = torch.Generator().manual_seed(21)
    args = [torch.randn(2, 9, 64, generator=g).to(dev) for _ in range(3)]
    args += [(0.3 * torch.randn(64, 1, 4, generator=g)).to(dev) for _ in range(3)]
    # fp32 sums of a few hundred terms, five in a row
    _check(canon_conv, lambda *a: tuple(_conv(x, w) for x, w in zip(a[:3], a[3:])), args, live, 1e-4)


@pytest.mark.parametrize("live", [(0,), (1,), (0, 1)])
def test_head_norm(dev, live):
    from atma_amd.kernel.train_glue import head_norm_train
    g = torch.Generator().manual_seed(22)
    args = [torch.randn(5, h, 64, generator=g).to(dev).bfloat16() for h in (4, 2)]
    w = [torch.randn(5, h, 64, generator=g).to(dev).bfloat16() for h in (4, 2)]

    def weigh(ys):   # (the norm of a normed row has no gradient)
        return tuple(y * t.to(y.dtype) for y, t in zip(ys, w))

    # bf16 results of first gradients that differ by a rounding or two, squared: as the MLP's double backward
    _check(lambda q, k: weigh(head_norm_train(q, k, 1e-6)),
           lambda q, k: weigh([F.rms_norm(t, (64,), eps=1e-6) for t in (q, k)]), args, live, 0.1)


@pytest.mark.parametrize("live", [(0,), (1,), (2, 3), (0, 1, 2, 3)])
def test_gate(dev, live):
    from atma_amd.kernel.train_glue import gate_train
    H, d, rows = 4, 64, 6
    g = torch.Generator().manual_seed(23)
    c = torch.randn(1, H, rows, d, generator=g)
    args = [t.to(dev).bfloat16() for t in (c, *(torch.randn(rows, H, d, generator=g) for _ in range(3)))]

    def eager(c, gate, r, mg):
        xa = c.transpose(1, 2).reshape(rows, H, d) * torch.sigmoid(gate)
        xm = F.rms_norm(r, (d,), eps=1e-6) * torch.sigmoid(mg)
        return torch.cat((xa.reshape(rows, -1), xm.reshape(rows, -1)), 1)

    _check(lambda c, gate, r, mg: gate_train(c.transpose(1, 2), gate, r, mg.reshape(rows, H * d), 1e-6), eager, args, live, 0.1)


@pytest.mark.parametrize("live", [(0,), (1, 3), (0, 2)])
def test_linears(dev, live):
    from atma_amd.kernel.train_glue import _LinearsFn
    g = torch.Generator().manual_seed(24)
    args = [torch.randn(7, 64, generator=g).to(dev).bfloat16()]
    args += [(64 ** -0.5 * torch.randn(n, 64, generator=g)).to(dev) for n in (32, 16)]
    args += [torch.randn(n, generator=g).to(dev) for n in (32, 16)]
    _check(lambda x, *p: _LinearsFn.apply(x, 0, False, *p),
           lambda x, w0, w1, b0, b1: (F.linear(x, w0, b0), F.linear(x, w1, b1)), args, live, 0.1)
