"""Training forms of the global block's projections, gates and MLP activation (16-bit rows on the GPU, fp32 or 16-bit
parameters): each one autograd node whose launches are the library GEMM and the kernels of ``train_glue.hip``.

Mirrors the eager math of ``model/reference.py:22-28`` (a Linear casts its parameters to the input's type),
``model/reference.py:127-195`` (projections, per-head norms, the gated output), ``model/blocks.py:472-490`` (the memory
readout's norm and gate) and ``model/layers.py:19-31`` (the MLP).  Every backward under ``create_graph`` differentiates
the eager form.  ``train_glue_served`` says where they apply; elsewhere the callers stay eager."""

import ctypes

import torch
import torch.nn.functional as F

from .. import _lib, _ops
from .layer_fusions import global_gate, head_rms_norm

_MAX = 16
_MAX_ROWS = 65535 * 128   # gather_colsum's grid
_P, _L, _I = ctypes.c_void_p * _MAX, ctypes.c_int64 * _MAX, ctypes.c_int32 * _MAX
_PLAIN = (torch.Tensor, torch.nn.Parameter)
_any_global_hook = torch.nn.modules.module._has_any_global_hook


def plain_module(m, cls):
    """``m`` is a ``cls`` itself (no subclass, no parametrisation, no ``forward`` of its own) and nothing hooks into its
    calls, or into every module's: a fused call may stand in for it."""
    if type(m) is not cls:
        return False
    own = m.__dict__
    return not (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"] or own["_backward_pre_hooks"]
                or "forward" in own or _any_global_hook())


def train_glue_served(x, *params):
    """Whether rows ``x`` with these parameters (None allowed) take the fused training forms: eager autograd on 16-bit
    GPU rows, parameters in fp32 or the rows' type at 16-byte aligned addresses (the kernels' loads; a view behind an odd
    offset of a flat buffer is not), nothing tracing, transforming or dispatching around it."""
    # what records the call first: a compiler refuses some of the questions after it
    if not torch.is_grad_enabled() or _ops.watched() or torch.is_autocast_enabled("cuda"):
        return False
    if not (x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and x.numel() > 0 and type(x) in _PLAIN
            and not x.is_inference() and x.numel() // x.shape[-1] <= _MAX_ROWS):
        return False
    return all(p is None or (type(p) in _PLAIN and not p.is_inference() and p.device == x.device and p.is_contiguous()
                             and p.dtype in (torch.float32, x.dtype) and p.shape[-1] % 8 == 0 and p.shape[0] % 8 == 0
                             and p.data_ptr() % 16 == 0)
               for p in params)


def _cast_blocks(blocks):
    """One launch of (src, dst, rows, cols, src_ld, dst_ld, sum, add) blocks."""
    n = len(blocks)
    code = _lib.dtype_code
    rc = _lib.load().atma_cast_blocks(
        n, _P(*[b[0].data_ptr() for b in blocks]), _P(*[_lib.ptr(b[7]) for b in blocks]),
        _P(*[b[1].data_ptr() for b in blocks]), _L(*[b[2] for b in blocks]), _L(*[b[3] for b in blocks]),
        _L(*[b[4] for b in blocks]), _L(*[b[5] for b in blocks]), _I(*[code(b[0].dtype) for b in blocks]),
        _I(*[code(b[1].dtype) for b in blocks]), _L(*[b[6] for b in blocks]), _lib.stream_handle(blocks[0][1].device))
    _lib.check(rc, "cast_blocks")


def _rows2d(t, rows):
    """(rows, width) with unit inner stride and 16-byte aligned rows, by a copy if need be."""
    return _ops._rows16(t.reshape(rows, -1))


def eager_grads(outs, ins, gs):
    """The gradients of eager outs with respect to ins, differentiable themselves; None where an input is None or takes no
    gradient (frozen parameters, rows that nothing trained leads to) or an output's gradient is None."""
    live = [(o, g) for o, g in zip(outs, gs) if g is not None and o.requires_grad]
    idx = [i for i, t in enumerate(ins) if t is not None and t.requires_grad]
    res = [None] * len(ins)
    if live and idx:
        got = torch.autograd.grad([o for o, _ in live], [ins[i] for i in idx], [g for _, g in live], create_graph=True,
                                  allow_unused=True)
        for i, g in zip(idx, got):
            res[i] = g
    return res


class _LinearsFn(torch.autograd.Function):
    """Several Linears as one GEMM.  ``cols`` False: of one input x (rows, K), outputs side by side; with ``inter`` the
    first is split by heads into two of that width, (rows, H, inter) each.  ``cols`` True: of inputs side by side in x,
    outputs summed.  params: the weights, then the biases (None allowed)."""

    @staticmethod
    def forward(ctx, x, inter, cols, *params):
        n = len(params) // 2
        ws, bs = params[:n], params[n:]
        rows = x.shape[0]
        if n == 1 and ws[0].dtype == x.dtype and (bs[0] is None or bs[0].dtype == x.dtype):
            w16, b16 = ws[0], bs[0]
        else:
            N = ws[0].shape[0] if cols else sum(w.shape[0] for w in ws)
            K = sum(w.shape[1] for w in ws) if cols else ws[0].shape[1]
            w16 = x.new_empty((N, K))
            b16 = x.new_empty(N) if any(b is not None for b in bs) else None
            blocks, at = [], 0
            for w, b in zip(ws, bs):
                dst = w16[:, at:] if cols else w16[at:]
                blocks.append((w, dst, w.shape[0], w.shape[1], w.shape[1], K, 1, None))
                if b is not None and not cols:
                    blocks.append((b, b16[at:], 1, b.shape[0], 0, 0, 1, None))
                elif b16 is not None and not cols:
                    b16[at:at + w.shape[0]].zero_()
                at += w.shape[1] if cols else w.shape[0]
            if cols and b16 is not None:   # one or two biases
                b = [t for t in bs if t is not None]
                blocks.append((b[0], b16, 1, N, 0, 0, 1, b[1] if len(b) > 1 else None))
            _cast_blocks(blocks)
        y = F.linear(x, w16, b16)
        ctx.inter, ctx.cols, ctx.n = inter, cols, n
        ctx.set_materialize_grads(False)
        # the parameters by reference, for their shapes and for create_graph: only the converted copy is needed otherwise, so
        # they may change before the backward, as they may when the conversion is an autograd node of its own
        ctx.params, ctx.versions = params, [None if p is None else p._version for p in params]
        ctx.save_for_backward(x, w16)
        if cols or (n == 1 and not inter):
            return y
        outs, at = [], 0
        for i, w in enumerate(ws):
            o = y[:, at:at + w.shape[0]]
            at += w.shape[0]
            if i == 0 and inter:
                o = o.view(rows, -1, 2, inter)
                outs += [o[:, :, 0], o[:, :, 1]]
            else:
                outs.append(o)
        return tuple(outs)

    @staticmethod
    def backward(ctx, *gs):
        x, w16 = ctx.saved_tensors
        params = ctx.params
        n, inter, rows = ctx.n, ctx.inter, x.shape[0]
        ws, bs = params[:n], params[n:]
        need = ctx.needs_input_grad
        if all(g is None for g in gs):
            return (None,) * len(need)
        if torch.is_grad_enabled():   # create_graph: the eager form
            if ctx.versions != [None if p is None else p._version for p in params]:
                raise RuntimeError("a parameter needed for the double backward has been modified by an inplace operation")
            return _linears_double(x, inter, ctx.cols, ws, bs, gs)
        widths = ([inter * (ws[0].shape[0] // (2 * inter))] * 2 if inter else []) + \
            [w.shape[0] for w in (ws[:1] if ctx.cols else ws[1 if inter else 0:])]
        parts = [None if g is None else _rows2d(g, rows) for g in gs]
        N = sum(widths)
        one = len(parts) == 1 and parts[0].is_contiguous()
        dy = parts[0] if one else x.new_empty((rows, N))
        lib = _lib.load()
        want_b = any(b is not None and need[3 + n + i] for i, b in enumerate(bs))
        if want_b or not one:
            part = torch.empty((lib.atma_gather_colsum_partials(rows), N), device=x.device, dtype=torch.float32)
            rc = lib.atma_gather_colsum(len(parts), _P(*[_lib.ptr(p) for p in parts]),
                                        _L(*[0 if p is None else p.stride(0) for p in parts]), _L(*widths), inter or 0,
                                        None if one else dy.data_ptr(), part.data_ptr(), rows,
                                        _lib.dtype_code(x.dtype), _lib.stream_handle(x.device))
            _lib.check(rc, "gather_colsum")
        dx = dy @ w16 if need[0] else None
        grads, blocks = [None] * (2 * n), []
        if any(need[3:3 + n]):
            dw = dy.t() @ x
            at = 0
            for i, w in enumerate(ws):
                if need[3 + i]:
                    if n == 1 and w.dtype == x.dtype:
                        grads[0] = dw
                    else:
                        grads[i] = torch.empty_like(w)
                        blocks.append((dw[:, at:] if ctx.cols else dw[at:], grads[i], w.shape[0], w.shape[1],
                                       dw.shape[1], w.shape[1], 1, None))
                at += w.shape[1] if ctx.cols else w.shape[0]
        at = 0
        for i, w in enumerate(ws):
            if bs[i] is not None and need[3 + n + i]:
                grads[n + i] = torch.empty_like(bs[i])
                blocks.append((part[:, at:], grads[n + i], 1, w.shape[0], N, 0, part.shape[0], None))
            at += 0 if ctx.cols else w.shape[0]
        if blocks:
            _cast_blocks(blocks)
        return (dx, None, None, *grads)


def _linears_double(x, inter, cols, ws, bs, gs):
    ws16, bs16 = [w.type_as(x) for w in ws], [None if b is None else b.type_as(x) for b in bs]
    if cols:
        ks = [w.shape[1] for w in ws]
        outs = [sum(F.linear(xi, w, b) for xi, w, b in zip(x.split(ks, 1), ws16, bs16))]
    else:
        outs = [F.linear(x, w, b) for w, b in zip(ws16, bs16)]
        if inter:
            o = outs[0].view(x.shape[0], -1, 2, inter)
            outs = [o[:, :, 0], o[:, :, 1]] + outs[1:]
    res = eager_grads(outs, [x, *ws, *bs], gs)
    return (res[0], None, None, *res[1:])


def linear_train(x, weight, bias):
    """``F.linear(x, weight.type_as(x), bias.type_as(x))``: one launch converts the parameters, the bias gradient is an
    fp32 column sum and one launch converts both gradients back."""
    y = _LinearsFn.apply(x.reshape(-1, x.shape[-1]), 0, False, weight, bias)
    return y.view(*x.shape[:-1], weight.shape[0])


def project_train(x, linears, head_dim):
    """The Linears of one input x (rows, K) as one GEMM: (the first's halves of every head, (rows, H, head_dim) each,
    then each other's (rows, N)), views of one buffer."""
    return _LinearsFn.apply(x, head_dim, False, *[m.weight for m in linears], *[m.bias for m in linears])


def out_train(x, linears):
    """The sum of two Linears whose inputs lie side by side in x (rows, K0 + K1), as one GEMM."""
    return _LinearsFn.apply(x, 0, True, *[m.weight for m in linears], *[m.bias for m in linears])


class _HeadNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, eps):
        ctx.eps = eps
        ctx.save_for_backward(q, k)
        return head_rms_norm(q, eps), head_rms_norm(k, eps)

    @staticmethod
    def backward(ctx, dq, dk):
        xs = ctx.saved_tensors
        if torch.is_grad_enabled():
            ys = [F.rms_norm(x, (x.shape[-1],), eps=ctx.eps) for x in xs]
            return (*eager_grads(ys, xs, (dq, dk)), None)
        rows, d = xs[0].shape[0], xs[0].shape[2]
        dn = [_ops._aligned16(g) for g in (dq, dk)]
        dx = [torch.empty_like(g) for g in dn]
        rc = _lib.load().atma_head_norm_bwd(
            _P(*[x.data_ptr() for x in xs]), _L(*[x.stride(0) for x in xs]), _L(*[x.stride(1) for x in xs]),
            _L(*[x.shape[1] for x in xs]), _P(*[g.data_ptr() for g in dn]), _P(*[g.data_ptr() for g in dx]), rows, d,
            float(ctx.eps), _lib.dtype_code(xs[0].dtype), _lib.stream_handle(xs[0].device))
        _lib.check(rc, "head_norm_bwd")
        return dx[0], dx[1], None


def head_norm_train(q, k, eps):
    """``F.rms_norm`` of every head of q (rows, H, d) and k (rows, Hkv, d), both read in place."""
    return _HeadNormFn.apply(q, k, eps)


class _GateFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, c, gate, r, mgate, eps):
        rows, H, d = gate.shape
        out = c.new_empty((rows, 2 * H * d))
        global_gate(c, gate, r, mgate, eps, out=out)
        ctx.eps = eps
        ctx.save_for_backward(c, gate, r, mgate)
        return out

    @staticmethod
    def backward(ctx, dx):
        c, gate, r, mgate = ctx.saved_tensors
        rows, H, d = gate.shape
        if torch.is_grad_enabled():
            xa = (c * torch.sigmoid(gate.view_as(c))).reshape(rows, H * d)
            xm = F.rms_norm(r, (d,), eps=ctx.eps).reshape(rows, H * d) * torch.sigmoid(mgate)
            return (*eager_grads([torch.cat((xa, xm), 1)], (c, gate, r, mgate), [dx]), None)
        dx = _ops._aligned16(dx)
        dc, dgate, dr, dmg = (c.new_empty((rows, H, d)) for _ in range(4))
        rc = _lib.load().atma_global_gate_bwd(
            c.data_ptr(), c.stride(0), c.stride(1), c.stride(2), c.shape[1], gate.data_ptr(), gate.stride(0),
            gate.stride(1), r.data_ptr(), mgate.data_ptr(), mgate.stride(0), dx.data_ptr(), dc.data_ptr(),
            dgate.data_ptr(), dr.data_ptr(), dmg.data_ptr(), rows, H, d, float(ctx.eps), _lib.dtype_code(c.dtype),
            _lib.stream_handle(c.device))
        _lib.check(rc, "global_gate_bwd")
        return dc.view(c.shape), dgate, dr, dmg.view(rows, H * d), None


def gate_train(c, gate, r, mgate, eps):
    """``global_gate``'s two projection inputs side by side (rows, 2 H d): c (B, T, H, d) view, gate (rows, H, d) view,
    r (rows, H, d) contiguous, mgate (rows, H d), all 16-bit of one type."""
    return _GateFn.apply(c, gate, r, mgate, eps)


class _SquaredReluGateFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y):
        ctx.save_for_backward(y)
        W = y.shape[1] // 2
        return _ops.run.squared_relu_gate(y[:, :W], y[:, W:])

    @staticmethod
    def backward(ctx, dh):
        y, = ctx.saved_tensors
        W = y.shape[1] // 2
        if torch.is_grad_enabled():
            a, gate = y.chunk(2, 1)
            return eager_grads([gate * a.relu().square()], [y], [dh])[0]
        dh = _rows2d(dh, y.shape[0])
        dy = torch.empty_like(y)
        rc = _lib.load().atma_squared_relu_gate_bwd(y.data_ptr(), y.stride(0), dh.data_ptr(), dh.stride(0), dy.data_ptr(),
                                                    y.shape[0], W, _lib.dtype_code(y.dtype),
                                                    _lib.stream_handle(y.device))
        _lib.check(rc, "squared_relu_gate_bwd")
        return dy


def squared_relu_gate_train(y):
    """``gate * relu(a)^2`` with y (rows, 2 W) contiguous = [a | gate]."""
    return _SquaredReluGateFn.apply(y)
