"""The serving prefills' recurrence, its states rows of a table advanced in place and its sequences ragged in one launch,
against the general call per sequence (gathered state in, final state out).  Both scan a sequence's chunks in the same
order with the same kernels, so they agree to the bit unless one of them splits the sequence along tokens."""

import pytest
import torch

from helpers import rel_err

pytestmark = pytest.mark.gpu

RAGGED = {
    "edges": [1, 0, 63, 64, 65, 129, 2],
    "many": [(37 * i) % 200 for i in range(70)],      # more than one launch's 64 sequences, some empty
    "one": [200],
    "long": [4160, 5, 300],                           # one far longer than the rest: split along tokens
}


def _inputs(dev, dtype, lens, H, Hkv, d, rows):
    g = torch.Generator().manual_seed(sum(lens) + d)
    t, mv = sum(lens), lambda x: x.to(dev)  # noqa: E731
    q = mv(torch.randn(t, H, d, generator=g).to(dtype))
    kv = mv(torch.randn(t, 2, Hkv, d, generator=g).to(dtype))        # k and v: strided views of one buffer
    zg, zb = mv(torch.randn(t, H, generator=g)), mv(torch.randn(t, H, generator=g))
    table = mv(torch.randn(rows, H, d, d, generator=g) * 0.1)
    slots = mv(torch.randperm(rows, generator=g)[:len(lens)])
    return q, kv[:, 0], kv[:, 1], zg, zb, table, slots


@pytest.mark.parametrize("lens", RAGGED)
@pytest.mark.parametrize("dtype,H,Hkv,d", [(torch.bfloat16, 8, 2, 128), (torch.float16, 4, 4, 64)])
@torch.no_grad()
def test_ragged_equals_one_by_one(dev, lens, dtype, H, Hkv, d):
    from atma_amd.kernel import chunk_gated_delta_rule
    from atma_amd.kernel.gated_delta import gated_delta_prefill
    lens = RAGGED[lens]
    q, k, v, zg, zb, table, slots = _inputs(dev, dtype, lens, H, Hkv, d, len(lens) + 3)
    got = table.clone()
    o = gated_delta_prefill(q, k, v, zg, zb, got, slots, (3.9, 0.1), lens)
    torch.cuda.synchronize()
    ref, start = table.clone(), 0
    for i, n in enumerate(lens):
        s = slice(start, start + n)
        start += n
        ro, S = chunk_gated_delta_rule(*(x[s][None] for x in (q, k, v, zg, zb)), scale=1.0, gate_bias=(3.9, 0.1),
                                       initial_state=table[slots[i:i + 1]], output_final_state=True,
                                       use_qk_l2norm_in_kernel=True)
        ref[slots[i]] = S[0]
        if n < 1500:   # the general call's plain scan too
            assert torch.equal(o[s], ro[0]) and torch.equal(got[slots[i]], S[0]), n
        elif n:        # both split it, into the same segments
            assert rel_err(o[s], ro[0]) <= 5e-3 and rel_err(got[slots[i]], S[0]) <= 5e-3, n
    rest = torch.ones(table.shape[0], dtype=torch.bool, device=dev)
    rest[slots] = False
    assert torch.equal(got[rest], table[rest])   # no other row is touched


@pytest.mark.parametrize("B,T", [(1, 100), (3, 65), (1, 3000)])   # plain, plain, split
@torch.no_grad()
def test_dense_equals_gathered_states(dev, B, T):
    from atma_amd.kernel import chunk_gated_delta_rule
    from atma_amd.kernel.gated_delta import gated_delta_prefill
    q, k, v, zg, zb, table, slots = _inputs(dev, torch.bfloat16, [T] * B, 8, 2, 128, B + 2)
    q, k, v, zg, zb = (x.unflatten(0, (B, T)) for x in (q, k, v, zg, zb))
    got = table.clone()
    slots[0] -= table.shape[0]     # a negative row counts from the end, as in an indexed read
    o = gated_delta_prefill(q, k, v, zg, zb, got, slots, (3.9, 0.1))
    ro, S = chunk_gated_delta_rule(q, k, v, zg, zb, scale=1.0, gate_bias=(3.9, 0.1), initial_state=table[slots],
                                   output_final_state=True, use_qk_l2norm_in_kernel=True)
    ref = table.clone()
    ref[slots] = S
    assert torch.equal(o, ro) and torch.equal(got, ref)
