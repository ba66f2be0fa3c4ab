"""The global layer's Canon step over whole rows, backed by libatma_hip.so (C ABI ``atma_canon_qkv``,
``atma_canon_bwd``): per-head RMSNorm of q and k and the residual causal depthwise convs of q, k and v
(``model/reference.py:136-155``), with the engine's conv tails (``inference/models/atma.py:102-162``) and the paged
KV write (``inference/layers/attention.py:7-56``) for the serving routes.

``canon_qkv`` is the inference form, one launch; ``canon_conv`` the differentiable convs alone (the norms stay torch
ops in training).  16-bit or fp32 GPU rows, head widths 64 and 128, kernel sizes 2 to 4.
"""

import ctypes

import torch
import torch.nn.functional as F

from .. import _lib, _ops  # noqa: F401  (_ops registers torch.ops.atma_hip.*)
from .train_glue import eager_grads

_DT = (torch.float32, torch.bfloat16, torch.float16)
_P3, _L3, _I3 = ctypes.c_void_p * 3, ctypes.c_int64 * 3, ctypes.c_int * 3


def canon_supported(x, head_dim, kernel_size):
    """True when the HIP Canon step serves rows like ``x`` (outside autocast, which would cast the eager conv)."""
    return (x.is_cuda and x.dtype in _DT and head_dim in (64, 128) and 2 <= kernel_size <= 4
            and not torch.is_autocast_enabled())


def _taps(weights, dtype):
    """Conv1d weights (C, 1, K) as contiguous aligned taps, all in the rows' dtype or all in fp32."""
    dt = torch.float32 if all(w.dtype == torch.float32 for w in weights) else dtype
    return [w if w.dtype == dt and w.is_contiguous() and w.data_ptr() % 16 == 0 else _ops._aligned16(w.detach().to(dt))
            for w in weights], dt


def _layout(xs):
    return [t.data_ptr() for t in xs], [t.stride(0) for t in xs], [t.stride(1) for t in xs]


@torch.no_grad()
def canon_qkv(q, k, v, weights, eps, *, seq_len=0, token_maps=None, tails=None, slots=None, continuing=False,
              caches=None, slot_mapping=None):
    """``x + conv(x)`` of v and of the per-head RMS-normed (``eps``) q and k, one launch.

    q: (rows, H, d), k, v: (rows, Hkv, d) views with unit inner stride, read in place where head-rows are 16-byte aligned
    (q as the first half of every head of the q|gate projection).  weights: the three depthwise conv weights.  Rows
    are sequences of ``seq_len``, or packed by ``token_maps`` (starts, ends, table rows; int32, one per token).
    ``tails``: the three conv state tables (rows, C, K - 1), written with each sequence's last K - 1 conv inputs in
    row ``slots[b]`` (or the token map's); ``continuing`` reads them first as the left context, and counts negative rows
    from the table's end as indexing does (a fresh sequence without a row, negative, keeps no tail).  ``caches`` (k, v)
    with ``slot_mapping`` int32: the k / v rows also go to the paged caches, slots < 0 skipped.
    Returns contiguous (rows, H, d), (rows, Hkv, d), (rows, Hkv, d)."""
    rows, H, d = q.shape
    xs, heads = (q, k, v), (H, k.shape[1], v.shape[1])
    taps, wdt = _taps(weights, q.dtype)
    K = taps[0].shape[-1]
    for t, h, w in zip(xs, heads, taps):
        if t.shape != (rows, h, d) or t.dtype != q.dtype or t.stride(2) != 1 or w.numel() != h * d * K:
            raise ValueError("canon_qkv: q, k, v (rows, heads, d) in one dtype and conv weights (heads d, 1, K)")
    ptrs, ldr, ldh = _layout(xs)
    if (ptrs[0] | ptrs[1] | ptrs[2] | (ldr[0] | ldr[1] | ldr[2] | ldh[0] | ldh[1] | ldh[2]) * q.element_size()) % 16:
        xs = [_ops._rows16(t) for t in xs]
        ptrs, ldr, ldh = _layout(xs)
    dev = q.device
    outs = [torch.empty((rows, h, d), device=dev, dtype=q.dtype) for h in heads]
    tp, ts, num_slots = (None,) * 3, (0,) * 3, 0
    if tails is not None:
        for t, h in zip(tails, heads):
            if t.shape[1:] != (h * d, K - 1) or t.dtype != q.dtype or not t.is_contiguous():
                raise ValueError("canon_qkv: tails must be contiguous (slots, C, K - 1) in the rows' dtype")
        tp, ts, num_slots = [t.data_ptr() for t in tails], [t.stride(0) for t in tails], min(t.shape[0] for t in tails)
    cp, total_slots = (None,) * 3, 0
    if caches is not None:
        assert slot_mapping.numel() == rows
        for t, h in zip(caches, heads[1:]):
            if t.shape[2:] != (h, d) or t.dtype != q.dtype or not t.is_contiguous():
                raise ValueError("canon_qkv: caches must be contiguous (pages, page_size, Hkv, d) in the rows' dtype")
        cp, total_slots = (None, caches[0].data_ptr(), caches[1].data_ptr()), caches[0].shape[0] * caches[0].shape[1]
        slot_mapping = slot_mapping.to(device=dev, dtype=torch.int32).contiguous()
    maps = (None, None, None)
    if token_maps is not None:
        maps = [t.to(device=dev, dtype=torch.int32).reshape(-1).contiguous() for t in token_maps]
        if any(m.numel() != rows for m in maps):
            raise ValueError("token maps must have one entry per token")
    elif slots is not None:
        slots = slots.to(device=dev, dtype=torch.int64).reshape(-1).contiguous()
        if seq_len < 1 or slots.numel() * seq_len != rows:
            raise ValueError("canon_qkv: one table row for each sequence of seq_len tokens")
    if rows == 0:
        return outs
    rc = _lib.load().atma_canon_qkv(
        _P3(*ptrs), _L3(*ldr), _L3(*ldh), _L3(*heads),
        _I3(1, 1, 0), _P3(*[w.data_ptr() for w in taps]), _P3(*[o.data_ptr() for o in outs]), _P3(*tp), _L3(*ts),
        _P3(*cp), 3, rows, 0 if token_maps is not None else int(seq_len), *[_lib.ptr(m) for m in maps],
        _lib.ptr(slots if token_maps is None else None), num_slots, 1 if continuing else 0,
        _lib.ptr(slot_mapping if caches is not None else None), total_slots, K, d, float(eps), _lib.dtype_code(wdt),
        _lib.dtype_code(q.dtype), _lib.stream_handle(dev))
    _lib.check(rc, "canon_qkv")
    written = [t for ts_ in (tails, caches) if ts_ is not None for t in ts_]
    if written:   # as the dispatcher does for ops that write their arguments
        torch.autograd.graph.increment_version(written)
    return outs


def _conv_torch(x, w):
    """``x + conv(x)`` over (B, T, C) in torch (double backward only)."""
    y = F.conv1d(F.pad(x.transpose(1, 2), (w.shape[-1] - 1, 0)), w.to(x.dtype), groups=x.shape[2])
    return x + y.transpose(1, 2)


class _CanonConvFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, wq, wk, wv):
        ctx.save_for_backward(q, k, v, wq, wk, wv)
        return tuple(_ops.run.canon_conv([q, k, v], [wq, wk, wv]))

    @staticmethod
    def backward(ctx, *gy):
        saved = ctx.saved_tensors
        if torch.is_grad_enabled():   # create_graph: differentiable ops
            return tuple(eager_grads([_conv_torch(x, w) for x, w in zip(saved[:3], saved[3:])], saved, gy))
        return tuple(_ops.run.canon_conv_bwd([g.contiguous() for g in gy], list(saved[:3]), list(saved[3:])))


def canon_conv(q, k, v, wq, wk, wv):
    """Differentiable ``x + conv(x)`` of q, k, v (B, T, C) with depthwise conv weights (C, 1, K): one launch forward,
    two backward (dx and the weights' partial sums, then their reduction; weight gradients are fp32 sums)."""
    return _CanonConvFn.apply(q.contiguous(), k.contiguous(), v.contiguous(), wq, wk, wv)
