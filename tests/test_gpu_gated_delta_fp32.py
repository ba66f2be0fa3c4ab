"""The fp32 recurrence on the fp32 matrix instruction where it can go wrong: chunk edges, grouped heads, rows at odd
strides and offsets, decays that empty or keep the state, write strengths of 0 and 1; against the fp64 oracle at the fp32
bound of the other tests (1e-4 of values of order one)."""

import pytest
import torch

from helpers import max_abs
from oracle import gated_delta as OG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 16, 17, 64, 127, 129, 321])
@pytest.mark.parametrize("H,Hkv,d", [(2, 2, 64), (4, 1, 128)])
@pytest.mark.parametrize("decay,beta", [(-30.0, 1.0), (0.0, 1.0), (-1.0, 0.0), (-0.05, 0.5)])
def test_fp32_edges(dev, T, H, Hkv, d, decay, beta):
    from atma_amd.kernel import chunk_gated_delta_rule
    g = torch.Generator().manual_seed(T + d)
    B = 2
    # rows of odd length one element into a buffer: no 16-byte alignment anywhere
    buf = torch.randn(B, T, H + 2 * Hkv, d + 3, generator=g)
    q, k, v = (t[..., 1:d + 1] for t in buf.split([H, Hkv, Hkv], dim=2))
    glog = decay * torch.rand(B, T, H, generator=g) if decay > -30 else torch.full((B, T, H), decay)
    bt = torch.full((B, T, H), beta)
    S0 = torch.randn(B, H, d, d, generator=g) * 0.1
    dbuf = buf.to(dev)
    dq, dk, dv = (t[..., 1:d + 1] for t in dbuf.split([H, Hkv, Hkv], dim=2))
    o, S = chunk_gated_delta_rule(dq, dk, dv, glog.to(dev), bt.to(dev), scale=1.0, initial_state=S0.to(dev),
                                  output_final_state=True, use_qk_l2norm_in_kernel=True)
    e = H // Hkv
    o_ref, S_ref = OG.chunk_gated_delta_rule(q.double(), k.double().repeat_interleave(e, 2), v.double().repeat_interleave(e, 2),
                                             glog.double(), bt.double(), scale=1.0, initial_state=S0.double(),
                                             output_final_state=True, use_qk_l2norm_in_kernel=True)
    assert max_abs(o.cpu(), o_ref) <= 1e-4 and max_abs(S.cpu(), S_ref) <= 1e-4
