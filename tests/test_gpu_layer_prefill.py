"""The small launches around the layer's prefill against the chains they replace: gate logits, widened Polar
parameters, the paged K/V concatenation, and the layer's unsummed output finished alone."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,H", [(1, 128, 1), (15, 256, 8), (16, 1024, 8), (17, 1024, 9), (333, 384, 16), (3000, 1024, 3)])
@pytest.mark.parametrize("bias", [True, False])
def test_memory_gate_logits(dt, M, K, H, bias):
    from atma_amd.kernel.layer_fusions import memory_gate_logits
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(1, M, K, generator=g).to("cuda", dt)
    w = [torch.randn(H, K, generator=g).to("cuda", dt) for _ in range(2)]
    b = [torch.randn(H, generator=g).to("cuda", dt) if bias else None for _ in range(2)]
    got = memory_gate_logits(x, w[0], b[0], w[1], b[1])
    for z, wi, bi in zip(got, w, b):
        ref = x.double() @ wi.double().t() + (0 if bi is None else bi.double())
        size = x.double().abs() @ wi.double().abs().t() + 1
        assert z.dtype == torch.float32 and z.shape == (1, M, H)
        assert ((z - ref).abs() <= 2.0 ** -24 * (K / 4 + 8) * size).all()    # an fp32 sum of K exact products


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,d", [(1, 64), (8, 128), (16, 64)])
def test_polar_params_widened(dt, H, d):
    from atma_amd.kernel.polar import _params
    ps = [torch.randn(H, d, device="cuda").to(dt)] + [torch.randn(H, device="cuda").to(dt) for _ in range(4)]
    for a, b in zip(_params(ps[0].device, *ps), ps):
        assert a.dtype == torch.float32 and a.is_contiguous() and torch.equal(a, b.float())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("page,cached,T", [(16, 1, 1), (16, 16, 5), (256, 700, 3), (32, 95, 300), (256, 2560, 1000)])
def test_paged_kv_concat(dt, page, cached, T):
    from atma_amd.kernel.layer_fusions import paged_kv_concat
    Hkv, d = 2, 64
    n = (cached + page - 1) // page
    pool = n + 3
    kc, vc = (torch.randn(pool, page, Hkv, d, device="cuda").to(dt) for _ in range(2))
    pages = torch.randperm(pool)[:n].int().cuda()
    kn, vn = (torch.randn(T, 3, Hkv, d, device="cuda").to(dt)[:, 1] for _ in range(2))
    kb, vb = paged_kv_concat(kc, vc, pages, cached, kn, vn)
    for out, cache, new in ((kb, kc, kn), (vb, vc, vn)):
        assert torch.equal(out, torch.cat([cache[pages.long()].reshape(-1, Hkv, d)[:cached], new]))


@pytest.mark.parametrize("M,D,mu", [(1, 8, None), (7, 1024, 8), (33, 520, 16), (9000, 1024, 8), (5, 4096, 4)])
@pytest.mark.parametrize("parts", [0, 3])
def test_partial_sums_alone(M, D, mu, parts):
    from atma_amd.kernel.decode_fusions import PartialSums
    dt = torch.bfloat16
    base = torch.randn(M, D, device="cuda").to(dt) if not parts else None
    p = torch.randn(parts, M, D, device="cuda") if parts else None
    biases = [torch.randn(D, device="cuda").to(dt) for _ in range(3)]
    mx = None if mu is None else torch.randn(M, mu, device="cuda").to(dt)
    mw = None if mu is None else torch.randn(D, mu, device="cuda").to(dt)
    ps = PartialSums(p, biases, mu_x=mx, mu_w=mw, dtype=dt, base=base)
    with torch.no_grad():
        out = ps.materialize()
    ref = (base.double() if parts == 0 else p.double().sum(0)) + sum(b.double() for b in biases)
    if mu is not None:
        ref = ref + mx.double() @ mw.double().t()
    # one rounding of an fp32 sum: half a unit of the result and fp32 noise on terms of about sqrt(mu) + parts
    assert out.dtype == dt and ((out - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -18).all()
    torch.testing.assert_close(out, ps.materialize(), rtol=2.0 ** -6, atol=2.0 ** -16)   # grad mode: the torch sum
