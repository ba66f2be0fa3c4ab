"""16-bit training of the recurrence with grouped KV heads, which the kernels read in place and whose gradients a launch
sums: against the same call with the heads expanded by torch, whose summed gradients it must equal up to one rounding."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,Hkv,d", [(1, 1, 4, 1, 64), (2, 65, 6, 2, 128), (1, 200, 8, 8, 128), (3, 130, 8, 2, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_grouped_equals_expanded(dev, B, T, H, Hkv, d, dtype):
    from atma_amd.kernel import chunk_gated_delta_rule
    g = torch.Generator().manual_seed(T + H)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    q, k, v = (rnd(B, T, h, d).to(dtype).to(dev) for h in (H, Hkv, Hkv))
    zg = torch.nn.functional.logsigmoid(rnd(B, T, H) + 3.9).to(dev)
    beta, do = torch.sigmoid(rnd(B, T, H)).to(dev), rnd(B, T, H, d).to(dtype).to(dev)

    def run(expand):
        x = [t.detach().clone().requires_grad_() for t in (q, k, v, zg, beta)]
        kk, vv = (t.repeat_interleave(H // Hkv, 2) if expand else t for t in x[1:3])
        o, _ = chunk_gated_delta_rule(x[0], kk, vv, x[3], x[4], scale=1.0, use_qk_l2norm_in_kernel=True)
        return [o] + list(torch.autograd.grad(o, x, do))

    for i, (got, ref) in enumerate(zip(run(False), run(True))):
        if i in (2, 3):   # dk, dv: the same shares in fp32, in another order, rounded once: 1 ulp of the result
            ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10) * ref.float().abs()
            tiny = 2.0 ** -16 * ref.float().abs().max()   # where the shares cancel: fp32 sums of H / Hkv of them
            assert ((got.float() - ref.float()).abs() <= ulp + tiny).all(), i
        else:
            assert torch.equal(got, ref), i
