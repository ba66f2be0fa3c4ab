"""The fused training forms of the projections, norms, gates and MLP activation against float64 autograd of the eager
form, next to the eager 16-bit form's own error: both round 16-bit results of the same products, so neither may be off
by more than the other plus one rounding of the largest value (2^-8 bf16, 2^-11 fp16)."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
EPS = torch.finfo(torch.float32).eps


def _check(fused, eager, args, dtype, seed=0, live=None):
    """fused / eager: args -> tuple of outputs; compares outputs and every argument's gradient."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def run(fn, xs):
        xs = [x.detach().clone().requires_grad_(x.is_floating_point()) for x in xs]
        outs = fn(*xs)
        outs = outs if isinstance(outs, tuple) else (outs,)
        return outs, xs

    o1, x1 = run(fused, args)
    o2, x2 = run(eager, args)
    o3, x3 = run(eager, [a.double() for a in args])
    use = range(len(o1)) if live is None else live
    ws = [torch.randn(o.shape, device="cuda", generator=g) for o in o1]
    res = []
    for outs, xs in ((o1, x1), (o2, x2), (o3, x3)):
        loss = [(outs[i], ws[i].to(outs[i].dtype)) for i in use]
        gr = torch.autograd.grad([o for o, _ in loss], xs, [w for _, w in loss], allow_unused=True)
        res.append([o.detach() for o in outs] + list(gr))
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for i, (a, b, c) in enumerate(zip(*res)):
        if c is None:   # an argument that no used output depends on: zeros or none
            assert a is None or not a.any(), i
            continue
        assert a.dtype == b.dtype and a.shape == b.shape, i
        ea, eb = (a.double() - c).abs().max().item(), (b.double() - c).abs().max().item()
        assert ea <= eb + unit * c.abs().max().item(), (i, ea, eb)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("wdt", [torch.float32, None])
@pytest.mark.parametrize("rows,K,outs,d", [(1, 8, (128, 8), 64), (129, 256, (512, 128, 128, 256, 8, 8), 128),
                                           (300, 64, (256, 264), 0), (257, 136, (72,), 0)])
def test_project(dev, dtype, wdt, rows, K, outs, d):
    from atma_amd.kernel.train_glue import _LinearsFn
    x = torch.randn(rows, K, device=dev).to(dtype)
    ws = [(torch.randn(n, K, device=dev) * K ** -0.5).to(wdt or dtype) for n in outs]
    bs = [torch.randn(n, device=dev).to(wdt or dtype) for n in outs]
    n = len(outs)

    def fused(x, *p):
        return _LinearsFn.apply(x, d, False, *p)

    def eager(x, *p):
        ys = [F.linear(x, w.type_as(x), b.type_as(x)) for w, b in zip(p[:n], p[n:])]
        if d:
            ys = list(ys[0].view(rows, -1, 2, d).unbind(2)) + ys[1:]
        return tuple(ys)

    _check(fused, eager, [x, *ws, *bs], dtype)
    if n > 1:
        _check(fused, eager, [x, *ws, *bs], dtype, live=[0])   # the other outputs' gradients are None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 130, 513])
def test_glue(dev, dtype, rows):
    from atma_amd.kernel.train_glue import gate_train, head_norm_train, out_train, squared_relu_gate_train
    H, Hkv = 6, 2
    for d in (64, 128):
        qg, k = (torch.randn(rows, h, w, device=dev).to(dtype) for h, w in ((H, 2 * d), (Hkv, d)))
        _check(lambda a, b: head_norm_train(a[..., :d], b, EPS),
               lambda a, b: tuple(F.rms_norm(t, (d,), eps=EPS) for t in (a[..., :d], b)), [qg, k], dtype)
        c, gate, r, mg = (torch.randn(rows, H, d, device=dev).to(dtype) for _ in range(4))
        c = c.view(1, rows, H, d).transpose(1, 2).contiguous()

        def eager(c, gate, r, mg):
            xa = c.transpose(1, 2).reshape(rows, H, d) * torch.sigmoid(gate)
            xm = F.rms_norm(r, (d,), eps=EPS) * torch.sigmoid(mg)
            return torch.cat((xa.reshape(rows, -1), xm.reshape(rows, -1)), 1)

        _check(lambda c, gate, r, mg: gate_train(c.transpose(1, 2), gate, r, mg.reshape(rows, H * d), EPS), eager,
               [c, gate, r, mg], dtype)
    y = torch.randn(rows, 2 * 72, device=dev).to(dtype)
    _check(squared_relu_gate_train, lambda y: y.chunk(2, 1)[1] * y.chunk(2, 1)[0].relu().square(), [y], dtype)
    lin = [torch.nn.Linear(k, 40, device=dev) for k in (128, 72)]
    x = torch.randn(rows, 200, device=dev).to(dtype)
    ps = [m.weight.detach() for m in lin] + [m.bias.detach() for m in lin]
    from atma_amd.kernel.train_glue import _LinearsFn
    _check(lambda x, *p: _LinearsFn.apply(x, 0, True, *p),
           lambda x, w0, w1, b0, b1: F.linear(x[:, :128], w0.type_as(x), b0.type_as(x)) +
           F.linear(x[:, 128:], w1.type_as(x), b1.type_as(x)), [x, *ps], dtype)
    assert out_train(x, lin).shape == (rows, 40)


def test_double_backward_frozen_and_hooks(dev):
    """create_graph differentiates the eager form; frozen parameters get no gradient; a hooked or traced Linear stays
    eager."""
    from atma_amd.kernel.train_glue import plain_module, train_glue_served
    from atma_amd.layers.global_attention import MLP, Linear
    torch.manual_seed(0)
    m = MLP(16).to(dev)
    m.fc.bias.requires_grad_(False)
    x = torch.randn(3, 5, 16, device=dev).bfloat16().requires_grad_()
    y = m(x)
    g, = torch.autograd.grad(y.float().square().sum(), x, create_graph=True)
    gg = torch.autograd.grad(g.float().square().sum(), [x, m.fc.weight, m.proj.weight])
    x2 = x.detach().float().requires_grad_()
    g2, = torch.autograd.grad(m(x2).square().sum(), x2, create_graph=True)
    ref = torch.autograd.grad(g2.square().sum(), [x2, m.fc.weight, m.proj.weight])
    for a, b in zip(gg, ref):
        assert (a.float() - b).abs().max() <= 0.1 * b.abs().max()    # bf16 through four GEMMs, against fp32
    y = m(x)
    with torch.no_grad():   # a parameter may change between forward and backward: its converted copy is what is saved
        m.proj.weight.mul_(1.0)
    y.float().sum().backward()
    assert m.fc.bias.grad is None and m.fc.weight.grad is not None and m.proj.bias.grad is not None
    odd = MLP(5).to(dev)   # widths that the launches do not serve: eager
    odd(torch.randn(3, 5, device=dev).bfloat16().requires_grad_()).float().sum().backward()
    lin = Linear(16, 16).to(dev)
    h = lin.register_forward_hook(lambda *a: None)
    assert not plain_module(lin, Linear)
    h.remove()
    assert plain_module(lin, Linear) and train_glue_served(x, lin.weight, lin.bias)
    with torch.autocast("cuda", torch.bfloat16):
        assert not train_glue_served(x, lin.weight, lin.bias)
    with torch.autograd.forward_ad.dual_level():
        assert not train_glue_served(x, lin.weight, lin.bias)
    assert torch.func.vmap(lin)(x.detach()).shape == x.shape
