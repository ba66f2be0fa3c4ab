"""Polar forward launches whose few tiles are split along the keys (chunk states merged by a second launch), against
the fp64 oracle: ragged tiles and chunks, windows, prefixes, rows without keys, fp32, and the saved statistics the
training backward reads."""

import pytest
import torch

from helpers import polar_params, rel_err
from oracle import polar as OP

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, Tq, Tk, d, dtype, window
    (1, 8, 2, 1500, 1500, 128, torch.bfloat16, None),
    (1, 8, 2, 2999, 2999, 128, torch.bfloat16, None),
    (1, 8, 2, 4000, 4000, 128, torch.bfloat16, 3000),
    (2, 4, 2, 1601, 1601, 64, torch.float16, None),
    (1, 8, 2, 300, 5003, 128, torch.bfloat16, None),     # a chunk behind a prefix
    (1, 2, 1, 1, 9000, 128, torch.float16, None),        # one row, many chunks
    (1, 8, 2, 300, 9000, 128, torch.bfloat16, 2500),     # ... with rows that need more blocks than the window's
    (1, 16, 4, 1429, 1429, 64, torch.bfloat16, None),
    (1, 8, 2, 1100, 1100, 128, torch.float32, None),
    (1, 8, 4, 130, 2500, 64, torch.float32, None),
    (2, 8, 8, 900, 900, 128, torch.float32, 600),
]


def _split_bytes(B, Hq, Hkv, Tq, Tk, d, dtype, causal, window):
    from atma_amd import _lib
    return _lib.load().atma_polar_attention_fwd_workspace_bytes(B, Hq, Hkv, Tq, Tk, d, _lib.dtype_code(dtype),
                                                                int(causal), window or 0)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(x).replace("torch.", "") for x in c))
def test_split_forward(case):
    from atma_amd.kernel import polar_attention_fwd
    B, Hq, Hkv, Tq, Tk, d, dtype, window = case
    assert _split_bytes(B, Hq, Hkv, Tq, Tk, d, dtype, Tq == Tk, window) > 0
    g = torch.Generator().manual_seed(Tq + Tk)
    q, k, v = (torch.randn(B, h, t, d, generator=g).to(dtype) for h, t in ((Hq, Tq), (Hkv, Tk), (Hkv, Tk)))
    p = polar_params(Hq, d, seed=4, prior=True)
    n = torch.arange(Tk - Tq + 1, Tk + 1, dtype=torch.float32)
    if Tq > 250 and Tq != Tk:
        n[7], n[140], n[200] = 0, 5, 64 * 9     # rows without keys, and within the first chunks
    c, m = polar_attention_fwd(q.cuda(), k.cuda(), v.cuda(), n.cuda(), is_causal=Tq == Tk, window=window,
                               **{a: t.cuda() for a, t in p.items()})
    rows = torch.tensor(sorted({0, 7, 63, 64, 127, 128, 140, 200, 255, 511, 512, 513, 640, Tq // 2, Tq - 2, Tq - 1}
                               & set(range(Tq))))
    cr, mr = OP.polar_rows(q.double(), k.double(), v.double(), n.double(), rows,
                           params={a: t.double() for a, t in p.items()}, window=window)
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    assert rel_err(c[:, :, rows.cuda()], cr) <= tol and rel_err(m[:, :, rows.cuda()], mr) <= tol
    assert torch.isfinite(c.float()).all() and torch.isfinite(m.float()).all()


@pytest.mark.parametrize("T,dtype", [(1200, torch.bfloat16), (900, torch.float32)])
def test_split_statistics_feed_the_backward(T, dtype):
    """Gradients through a split forward against fp64 autograd."""
    from atma_amd.kernel import polar_attention
    Hq, Hkv, d = 4, 2, 64
    assert _split_bytes(1, Hq, Hkv, T, T, d, dtype, True, None) > 0
    g = torch.Generator().manual_seed(T)
    ins = [torch.randn(1, h, T, d, generator=g).to(dtype) for h in (Hq, Hkv, Hkv)]
    p = polar_params(Hq, d, seed=5, prior=True)
    gc, gm = torch.randn(1, Hq, T, d, generator=g).to(dtype), torch.randn(1, Hq, T, generator=g).to(dtype)
    n = torch.arange(1, T + 1, dtype=torch.float32)
    dev = [t.cuda().requires_grad_(True) for t in ins]
    pd = {a: t.cuda().requires_grad_(True) for a, t in p.items()}
    out = polar_attention(*dev, n.cuda(), **pd)
    got = torch.autograd.grad(out, dev + list(pd.values()), [gc.cuda(), gm.cuda()])
    ref = [t.double().requires_grad_(True) for t in ins]
    pr = {a: t.double().requires_grad_(True) for a, t in p.items()}
    exact = torch.autograd.grad(OP.polar_online(*ref, n.double(), params=pr), ref + list(pr.values()),
                                [gc.double(), gm.double()])
    for a, b in zip(got, exact):
        assert rel_err(a, b) <= (1e-3 if dtype == torch.float32 else 5e-2)
