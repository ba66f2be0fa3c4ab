"""The segments' entry states of the split recurrence (few heads, long sequences), whose products run on the fp32 matrix
instruction: against the fp64 oracle under a decay so slow that every segment's state reaches the last token."""

import pytest
import torch

from helpers import rel_err
from oracle import gated_delta as OG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("T", [1024, 1536, 2500, 9000])   # 1, 3, 5 and 16 (d 64) or 13 segments, ragged
@pytest.mark.parametrize("state", [False, True])
def test_entry_states_carry_through_segments(dev, d, T, state):
    from atma_amd.kernel import chunk_gated_delta_rule
    gen = torch.Generator().manual_seed(T + d)
    B, H = 2, 2
    q, k, v = (torch.randn(B, T, H, d, generator=gen).bfloat16() for _ in range(3))
    glog = -1e-4 * torch.rand(B, T, H, generator=gen)
    beta = 0.05 * torch.rand(B, T, H, generator=gen)     # weak writes: the initial state survives as well
    S0 = torch.randn(B, H, d, d, generator=gen) if state else None
    o, S = chunk_gated_delta_rule(q.to(dev), k.to(dev), v.to(dev), glog.to(dev), beta.to(dev), scale=1.0,
                                  initial_state=None if S0 is None else S0.to(dev), output_final_state=True,
                                  use_qk_l2norm_in_kernel=True)
    # the same sequences among 16: heads enough for the plain scan, which has no entry states
    po, pS = chunk_gated_delta_rule(*(x.to(dev).repeat(8, *[1] * (x.dim() - 1)) for x in (q, k, v, glog, beta)), scale=1.0,
                                    initial_state=None if S0 is None else S0.to(dev).repeat(8, 1, 1, 1),
                                    output_final_state=True, use_qk_l2norm_in_kernel=True)
    o_ref, S_ref = OG.chunk_gated_delta_rule(q.double(), k.double(), v.double(), glog.double(), beta.double(), scale=1.0,
                                             initial_state=None if S0 is None else S0.double(), output_final_state=True,
                                             use_qk_l2norm_in_kernel=True)
    for got, plain, ref in ((o, po[:B], o_ref), (S, pS[:B], S_ref)):
        e, p = rel_err(got.cpu(), ref), rel_err(plain.cpu(), ref)
        # the file's bound for 16-bit rows, and the plain scan's own error with room for another order of rounding
        assert e <= 2e-2 and e <= 2 * p + 1e-3, (e, p)
