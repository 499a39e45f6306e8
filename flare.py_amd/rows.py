"""fp32 training of the token-wise layers (ResidualMLP, norms) over long row arrays: the library's products with HIP row passes
around them.

What torch runs as separate layers (pdebench/models/flare.py:45-59, 204-215) spends most of an fp32 training step outside the
products: in the backward the activation, the bias gradients and the sums at the residuals each make passes of their own over
[T,C], and the norms run far from the memory's rate.  Here a layer's backward is one pass over the rows (flare_rows_layer_bwd:
slope, both products and the bias sums); at the widths that kernel does not take, a pass that forms dt, the bias gradient and the
start value of dx together (flare_rows_act_bwd), the product that adds W^T dt to it, and the sliced weight gradient.  The norms are
one pass each way.

Used where the modules' fp32 Linear layers already run as a once-differentiable function (gradients enabled, outside autocast,
4096 rows or more) and the arrays are large enough (MIN_ELEMS); every other call keeps the torch layers.
"""
from __future__ import annotations

import ctypes as C

import torch
from torch import nn
from torch.nn.modules import module as _module
from torch.autograd.function import once_differentiable

from . import _lib, fused
from .functional import _on_device, _ptr, _stream_ptr

LONG_ROWS = 4096      # rows from which the modules' fp32 Linear layers slice their weight gradient (below, one product is as fast)
# Elements of a row array from which these nodes are used, at the widths whose layer backward is one pass (_ONE_PASS).  A layer enqueues
# less than torch's own nodes there, so they are faster at every size that was measured; a sequence block's step, torch's nodes / these,
# us: 64 channels, 8192 rows (0.5 Mi) 3047 / 2298, 16,384 rows 3066 / 2259, 98,304 rows (6 Mi) 3083 / 2273, 131,072 rows 3846 / 2341; 128
# channels, 8192 rows (1 Mi) 2946 / 2122, 65,536 rows 3176 / 2173, 131,072 rows 5548 / 3869.  The line is no break-even, then: it leaves
# arrays of 0.5 Mi elements and less on the torch layers, where they always were.  The other widths keep the separate passes, which
# enqueue a little more than torch's nodes do: there the line is 6 Mi, where a step waits for the kernels.  A step recorded into a graph
# has no host to wait for, but follows the same rule: its replays give the results of the eager step bit for bit.
MIN_ELEMS = 5 << 17
_ONE_PASS = (64, 128)
_WIDTHS = (32, 64, 128, 256)


def weight_grad(dy2, x2):
    """dY^T X over long rows as a batched product over slices (one product runs without splitting that axis)."""
    T = x2.shape[0]
    S = next(s for s in (64, 32, 16, 8, 4, 2, 1) if T % s == 0)
    if S > 1:
        return torch.bmm(dy2.view(S, T // S, -1).transpose(1, 2), x2.view(S, T // S, -1)).sum(0)
    return dy2.t() @ x2


def _plain(m):
    """No hooks, its own or global ones, and no forward replaced on the instance: its class's forward is all that calling it does."""
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or "forward" in m.__dict__
                or _module._has_any_global_hook())


def _param_ok(p):
    return p is None or (type(p) in (torch.Tensor, nn.Parameter) and p.is_cuda and p.dtype is torch.float32 and p.is_contiguous()
                         and p.data_ptr() % 16 == 0)


def _call_ok(x, long_rows):
    return (torch.is_grad_enabled() and type(x) in (torch.Tensor, nn.Parameter) and x.is_cuda and x.dtype is torch.float32
            and x.shape[-1] in _WIDTHS and x.numel() // x.shape[-1] >= long_rows and not torch.is_autocast_enabled()
            and x.numel() >= (MIN_ELEMS if x.shape[-1] in _ONE_PASS else MIN_ELEMS * 48 // 5)      # 6 Mi
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def chain_info(mod, x, long_rows=LONG_ROWS):
    """fused._layers_of(mod) where chain() takes the call, else None: square nn.Linear layers of x's width whose weights all ask
    for gradients, tanh-GELU or SiLU between them."""
    if not _call_ok(x, long_rows):
        return None
    info = fused._layers_of(mod)
    if info is None:
        return None
    width = x.shape[-1]
    for l in info[0]:
        if not (type(l) is nn.Linear and _plain(l) and l.in_features == width == l.out_features and l.weight.requires_grad
                and _param_ok(l.weight) and _param_ok(l.bias)):
            return None
    act = getattr(mod, "act", None)
    if act is not None and not (type(act) in (nn.GELU, nn.SiLU) and _plain(act)):
        return None
    return info


def _rows(t, width):
    """[T,C] contiguous fp32 rows on the 16-byte grid."""
    t2 = t.reshape(-1, width)
    if t2.dtype is not torch.float32:
        t2 = t2.float()
    if not t2.is_contiguous():
        t2 = t2.contiguous()
    return t2 if t2.data_ptr() % 16 == 0 else t2.clone()


def _parts(T, width):
    n = C.c_int32(0)
    _lib.check(_lib.load().flare_rows_parts(T, width, C.byref(n)), "flare_rows_parts")
    return n.value


def _layer_parts(T, width):
    """Partial results of flare_rows_layer_bwd, 0 where the separate passes serve the width."""
    n = C.c_int32(0)
    if width in _ONE_PASS:
        _lib.check(_lib.load().flare_rows_layer_bwd_parts(T, width, C.byref(n)), "flare_rows_layer_bwd_parts")
    return n.value


class _LinearLongRowsPass(torch.autograd.Function):
    """[res +] ([x +] act(x W^T + b)); inputs (act or -1, add, x, w, b, res).  One node per layer, as with torch's layers, and
    the forward gives their values bit for bit: a chain's outputs do not depend on whether a call comes here (a norm's in front of it
    do, in rounding: _NormFn reduces in an order of its own)."""

    @staticmethod
    def forward(ctx, act, add, x, w, b, res):
        width = x.shape[-1]
        s = _rows(x, width)
        t = torch.nn.functional.linear(s, w, b)
        if act == 0 or (act < 0 and add and res is not None):      # the activation and the sums in one pass
            r = None if res is None else _rows(res, width)
            y = torch.empty_like(t) if act == 0 else t
            with _on_device(t.device):
                rc = _lib.load().flare_rows_act_fwd(t.shape[0], width, act, _ptr(t), _ptr(s) if add else None, _ptr(r), _ptr(y),
                                                    C.c_void_p(_stream_ptr(t.device)))
            _lib.check(rc, "flare_rows_act_fwd")
            y = y.view(x.shape)
        else:
            y = t if act < 0 else torch.nn.functional.silu(t)
            if add:
                y = s + y
            y = y.view(x.shape)
            if res is not None:
                y = res + y
        ctx.act, ctx.add = act, add
        ctx.save_for_backward(s, w, t if act >= 0 else None)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        s, w, t = ctx.saved_tensors                          # through saved-tensor hooks in any memory order
        s, t = _rows(s, s.shape[-1]), None if t is None else _rows(t, t.shape[-1])
        act, T, width, dev = ctx.act, s.shape[0], s.shape[1], s.device
        _, _, need_x, need_w, need_b, need_res = ctx.needs_input_grad
        ds = _rows(dy, width)
        w = w.contiguous()
        parts = _layer_parts(T, width) if need_w and w.data_ptr() % 16 == 0 else 0
        if parts:
            dx = torch.empty_like(ds) if need_x else None
            part = torch.empty(parts, width + 1, width, dtype=torch.float32, device=dev)
            dw = torch.empty(width, width, dtype=torch.float32, device=dev)
            db = torch.empty(width, dtype=torch.float32, device=dev) if need_b else None
            at = part.data_ptr()
            with _on_device(dev):
                rc = _lib.load().flare_rows_layer_bwd(T, width, act, ctx.add, _ptr(ds), _ptr(t), _ptr(s), _ptr(w), _ptr(dx), at, at + 4 * parts * width * width,
                                                      _ptr(dw), _ptr(db), C.c_void_p(_stream_ptr(dev)))
            _lib.check(rc, "flare_rows_layer_bwd")
            return None, None, None if dx is None else dx.view(dy.shape), dw, db, dy if need_res else None
        dt = torch.empty_like(ds) if act >= 0 else ds
        dx = torch.empty_like(ds) if ctx.add and need_x else None
        db = torch.empty(width, dtype=torch.float32, device=dev) if need_b else None
        if act >= 0 or need_b or dx is not None:
            part = torch.empty(_parts(T, width), width, dtype=torch.float32, device=dev)
            with _on_device(dev):
                rc = _lib.load().flare_rows_act_bwd(T, width, act, _ptr(ds), _ptr(t), _ptr(dt) if act >= 0 else None, _ptr(dx), _ptr(part), _ptr(db),
                                                    C.c_void_p(_stream_ptr(dev)))
            _lib.check(rc, "flare_rows_act_bwd")
        dw = weight_grad(dt, s) if need_w else None
        if need_x:
            dx = dt @ w if dx is None else dx.addmm_(dt, w)
        return None, None, None if dx is None else dx.view(dy.shape), dw, db, dy if need_res else None


def chain(mod, x, info, res=None):
    """[res +] mod(x) for a call chain_info() accepts."""
    layers, act_mask, add_mask, act = info
    last = len(layers) - 1
    for i, l in enumerate(layers):
        x = _LinearLongRowsPass.apply(act if (act_mask >> i) & 1 else -1, bool((add_mask >> i) & 1), x, l.weight, l.bias,
                                      res if i == last else None)
    return x


def res_ok(res, x):
    return type(res) in (torch.Tensor, nn.Parameter) and res.dtype is torch.float32 and res.shape == x.shape and res.device == x.device


class _NormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, kind, eps, x, gamma, beta):
        x2 = _rows(x, x.shape[-1])
        y, stats = torch.empty_like(x2), torch.empty(x2.shape[0], 2, dtype=torch.float32, device=x.device)
        with _on_device(x.device):
            rc = _lib.load().flare_rows_norm_fwd(x2.shape[0], x2.shape[1], kind, eps, _ptr(x2), _ptr(gamma), _ptr(beta), _ptr(y), _ptr(stats),
                                                 C.c_void_p(_stream_ptr(x.device)))
        _lib.check(rc, "flare_rows_norm_fwd")
        ctx.kind = kind
        ctx.save_for_backward(x2, stats, gamma)
        return y.view(x.shape)

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        x2, stats, gamma = ctx.saved_tensors
        x2, stats = _rows(x2, x2.shape[-1]), stats.contiguous()
        T, width = x2.shape
        need = ctx.needs_input_grad            # (kind, eps, x, gamma, beta)
        dx = torch.empty_like(x2)
        part = torch.empty(_parts(T, width), 2, width, dtype=torch.float32, device=dy.device)
        gb = torch.empty(2, width, dtype=torch.float32, device=dy.device)
        dy2 = _rows(dy, width)
        with _on_device(dy.device):
            rc = _lib.load().flare_rows_norm_bwd(T, width, ctx.kind, _ptr(dy2), _ptr(x2), _ptr(stats), _ptr(gamma), None, _ptr(dx), _ptr(part),
                                                 _ptr(gb), C.c_void_p(_stream_ptr(dy.device)))
        _lib.check(rc, "flare_rows_norm_bwd")
        return None, None, dx.view(dy.shape) if need[2] else None, gb[0] if need[3] else None, gb[1] if need[4] else None


def norm(mod, x):
    """mod(x) for a nn.LayerNorm / nn.RMSNorm over the rows of x that a chain_info() chain reads next."""
    kind = {nn.LayerNorm: 1, nn.RMSNorm: 2}.get(type(mod))
    gamma, beta = getattr(mod, "weight", None), getattr(mod, "bias", None)
    if (kind is None or not _call_ok(x, LONG_ROWS) or not _plain(mod) or tuple(mod.normalized_shape) != (x.shape[-1],)
            or not _param_ok(gamma) or not _param_ok(beta)):
        return mod(x)
    eps = mod.eps if mod.eps is not None else torch.finfo(x.dtype).eps
    return _NormFn.apply(kind, float(eps), x, gamma, beta)
