"""The fused Canon step (``canon_qkv``, ``canon_conv``) against the chain it replaces in 64-bit torch: head norms,
residual causal convs, stored tails, cache rows and gradients, at strip edges, short chunks and every tap count."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
EPS = torch.finfo(torch.float32).eps
UNIT = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}  # unit roundoff: 2 ** -(significand bits)


def _conv64(x, w, left):
    """x + conv(x) of one sequence x (T, C) behind left (K - 1, C); and the same sum of magnitudes."""
    K = w.shape[-1]
    full = torch.cat([left, x])
    taps = [full[j:j + x.shape[0]] * w[:, 0, j] for j in range(K)]
    return x + sum(taps), x.abs() + sum(t.abs() for t in taps), full[full.shape[0] - (K - 1):]


def _inputs(g, rows, H, KV, d, dt, K, wdt):
    r = lambda *s, dtype=dt: torch.randn(*s, generator=g).to("cuda", dtype)  # noqa: E731
    qg = r(rows, H, 2 * d)
    return qg[..., :d], r(rows, KV, d), r(rows, KV, d), [r(h * d, 1, K, dtype=wdt) * 0.3 for h in (H, KV, KV)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d,H,KV,K,lens", [
    (128, 8, 2, 4, [1]), (128, 4, 1, 4, [2, 1, 3]), (64, 3, 2, 3, [9, 7]), (64, 16, 4, 4, [33, 32, 31]),
    (128, 2, 1, 2, [70]), (128, 8, 2, 4, [1000, 1200]), (128, 8, 2, 3, [3000] * 6)])
@pytest.mark.parametrize("mode", ["dense", "continuing", "packed"])
def test_canon_qkv(dt, d, H, KV, K, lens, mode):
    from atma_amd.kernel.canon import canon_qkv
    g = torch.Generator().manual_seed(len(lens) + d + K)
    if mode != "packed":
        lens = [lens[0]] * len(lens)
    rows, B = sum(lens), len(lens)
    q, k, v, ws = _inputs(g, rows, H, KV, d, dt, K, dt)
    heads = (H, KV, KV)
    tails = [torch.randn(B + 2, h * d, K - 1, generator=g).to("cuda", dt) for h in heads]
    old = [t.clone() for t in tails]
    slots = torch.randperm(B + 2, generator=g)[:B].cuda()
    pages = (rows + 15) // 16 + 1
    caches = [torch.zeros(pages, 16, KV, d, device="cuda", dtype=dt) for _ in range(2)]
    where = torch.randperm(pages * 16, generator=g)[:rows].int()
    where[::5] = -1
    kw = dict(seq_len=lens[0], slots=slots, continuing=mode == "continuing")
    if mode == "packed":
        n = torch.tensor(lens)
        ends = n.cumsum(0)
        kw = dict(token_maps=[t.repeat_interleave(n).int().cuda() for t in (ends - n, ends, slots.cpu())])
    outs = canon_qkv(q, k, v, ws, EPS, tails=tails, caches=caches, slot_mapping=where.cuda(), **kw)
    for i, (x, w, h) in enumerate(zip((q, k, v), ws, heads)):
        xn = x.double()
        if i < 2:
            xn = (xn * torch.rsqrt(xn.square().mean(-1, keepdim=True) + EPS)).to(dt).double()
        xn, at = xn.reshape(rows, h * d), 0
        for b, n in enumerate(lens):
            left = old[i][slots[b]].double().t() if mode == "continuing" else xn.new_zeros(K - 1, h * d)
            ref, mag, tail = _conv64(xn[at:at + n], w.double(), left)
            got = outs[i].view(rows, h * d)[at:at + n].double()
            # the norm may round to the neighbour of the 64-bit norm's rounding (two units of each term), the fp32
            # sums of K + 1 terms and the output round once more
            bound = (2 * UNIT[dt] + 16 * 2.0 ** -24) * mag + UNIT[dt] * ref.abs() + 1e-30
            assert ((got - ref).abs() <= 1.01 * bound).all(), (i, b)
            assert ((tails[i][slots[b]].double().t() - tail).abs() <= (2 * UNIT[dt] + 2.0 ** -21) * tail.abs()).all()
            at += n
        rest = [r for r in range(B + 2) if r not in slots.tolist()]
        assert torch.equal(tails[i][rest], old[i][rest])
    for c, o in zip(caches, outs[1:]):
        ref = torch.zeros_like(c).view(-1, KV, d)
        keep = (where >= 0).cuda()
        ref[where.cuda()[keep].long()] = o[keep]
        assert torch.equal(c.view(-1, KV, d), ref)


@pytest.mark.parametrize("dt,wdt", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16),
                                    (torch.float32, torch.float32)])
@pytest.mark.parametrize("B,T,C,K", [(1, 1, (64, 64, 128), 4), (3, 2, (256, 64, 64), 4), (2, 33, (512, 128, 128), 3),
                                     (3, 1031, (1024, 256, 256), 4), (1, 100, (128, 64, 64), 2)])
def test_canon_conv_gradients(dt, wdt, B, T, C, K):
    from atma_amd.kernel.canon import canon_conv
    g = torch.Generator().manual_seed(T)
    xs = [torch.randn(B, T, c, generator=g).to("cuda", dt).requires_grad_(True) for c in C]
    ws = [(torch.randn(c, 1, K, generator=g) * 0.3).to("cuda", wdt).requires_grad_(True) for c in C]
    gy = [torch.randn(B, T, c, generator=g).to("cuda", dt) for c in C]
    outs = canon_conv(*xs, *ws)
    grads = torch.autograd.grad(outs, xs + ws, gy)
    for i in range(3):
        x, w = xs[i].detach().double().requires_grad_(True), ws[i].detach().double().requires_grad_(True)
        y = x + F.conv1d(F.pad(x.transpose(1, 2), (K - 1, 0)), w, groups=C[i]).transpose(1, 2)
        gx, gw = torch.autograd.grad(y, (x, w), gy[i].double())
        for got, ref, u in ((outs[i], y.detach(), UNIT[dt]), (grads[i], gx, UNIT[dt]), (grads[3 + i], gw, UNIT[wdt])):
            # one rounding of an fp32 sum: of K + 1 terms, or for a weight of B T terms in strips of 32
            tol = 2 * u + (2.0 ** -24) * (64 + B * T / 32)
            assert ((got.double() - ref).norm() <= tol * ref.norm() * 1.5), i
