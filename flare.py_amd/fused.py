"""Fused path for the token-wise layers around the mixer (HIP kernels flare_mlp_fwd / flare_mlp_bwd).

`fused_mlp(x, mlp, norm=..., res=...)` evaluates, in ONE launch and without leaving the chip
between layers, what the reference runs as separate torch layers:

    res + ResidualMLP(norm(x))         pdebench/models/flare.py:45-59 and 204-215
    res + Linear(x)                    (out_proj, flare.py:156)

    ResidualMLP(in_dim <= 4, C, C)     (the models' in_proj, flare.py:137-140: the narrow first layer runs on
    ResidualMLP(C, C, out_dim <= 4)     the vector ALU; of out_proj's last layer only the real rows are stored)

A ResidualMLP with num_layers == 0 and a hidden width of E*C (2 <= E <= 8; the "4x expansion" feed-forward
block) runs in the same launch as E pairs of C x C tiles, the hidden activations never leaving the registers.

It is used by the modules only when the products may run in bf16/f16 (torch.autocast is on, or the
weights already are bf16/f16) — the conditions under which torch itself would run these Linear layers
in that type.  Everything else stays with the torch layers.  The 16-bit copies of the weights are
cached per module and rebuilt when a parameter changes.

With gradients enabled the chain of C x C layers (the k/v projections, the feed-forward block and the output
projection of a FLAREBlock at the reference's default ratios) runs through `_FusedMlpFn`: the same forward
launch, and a backward that recomputes the chain per token tile in one launch (flare_mlp_bwd) and forms the
parameter gradients from the rows it leaves with one more launch (flare_mlp_wgrad); the expanding two-layer MLP has a
backward launch of its own (flare_mlp_expand_bwd).  A stack with a narrow first input or last output runs that one
layer in a launch of its own while gradients are enabled and sends the C x C layers between through the same path.
Head-padded rows (narrow heads) have a backward in the few-token launches.
"""
from __future__ import annotations

import ctypes as C

import torch
from torch import nn
from torch.autograd.function import once_differentiable

from . import _lib
from .functional import _DTYPES, _autocast_dtype, _dtype_code, _on_device, _ptr, _stream_ptr

_SUPPORTED_C = (32, 64, 128)
_ACTS = {"gelu": 0, "silu": 1}


def _structure_key(mod):
    """Identity of everything the structural caches are built from: the layers, the activation module and the flags
    that set the masks.  Assigning a new submodule (a LoRA wrap, a re-initialisation by assignment) changes it: modules compare by
    identity, and a cache that keeps them, and not their ids, keeps another module from getting the id of one it was built from.
    Read from the module's own tables: every fused call asks several times, and attribute access on a Module goes
    through its __getattr__ for submodules."""
    if isinstance(mod, _SubChain):
        return None
    d = mod.__dict__
    nl = d.get("num_layers")
    if isinstance(mod, nn.Linear) or nl is None:
        return (type(mod),)
    m = d["_modules"]
    if nl == -1:
        return (-1, m["fc"], bool(d["residual"]))
    act = m["act"] if "act" in m else d.get("act")
    return (nl, m["fc1"], (*m["fcs"]._modules.values(),), m["fc2"], act,
            getattr(act, "approximate", None), bool(d["input_residual"]), bool(d["output_residual"]))


def _layers_of(mod):
    """(linear layers, act_mask, add_mask, act code) of a ResidualMLP or nn.Linear, or None.  The answer is kept on
    the module together with the submodules it was read from, and rebuilt when one of them is
    replaced."""
    key = _structure_key(mod)
    cached = mod.__dict__.get("_flare_layers")
    if cached is not None and cached[1] == key:
        return cached[0]
    info = _layers_of_uncached(mod)
    mod.__dict__["_flare_layers"] = (info, key)
    return info


def _layers_of_uncached(mod):
    if isinstance(mod, nn.Linear):
        return [mod], 0, 0, 0
    if getattr(mod, "num_layers", None) is None:
        return None
    if mod.num_layers == -1:
        return [mod.fc], 0, (1 if mod.residual else 0), 0
    layers = [mod.fc1, *mod.fcs, mod.fc2]
    L = len(layers)
    act_mask = (1 << (L - 1)) - 1
    add_mask = ((1 << (L - 1)) - 2) | (1 if mod.input_residual else 0) | ((1 << (L - 1)) if mod.output_residual else 0)
    if isinstance(mod.act, nn.GELU) and mod.act.approximate == "tanh":
        act = 0
    elif isinstance(mod.act, nn.SiLU):
        act = 1
    else:
        return None
    return layers, act_mask, add_mask, act


def _expand_factor(mod, Cdim):
    """E when mod is the two-layer MLP C -> E*C -> C (ResidualMLP with num_layers == 0 and no residual that
    applies), else 0."""
    if getattr(mod, "num_layers", None) != 0 or mod.input_residual or mod.output_residual:
        return 0
    f1, f2 = mod.fc1, mod.fc2
    hid = f1.out_features
    if f1.in_features != Cdim or f2.out_features != Cdim or f2.in_features != hid or hid % Cdim or hid == Cdim:
        return 0
    E = hid // Cdim
    return E if 2 <= E <= 8 else 0


def _io_dims(mod, layers):
    """(C, in_dim, out_dim) of a stack that is C x C except for a narrow (<= 4) first input and/or last output
    (0 = that end is C wide), or None."""
    if len(layers) < 2:
        return None
    Cdim = layers[0].out_features
    if any(l.in_features != Cdim or l.out_features != Cdim for l in layers[1:-1]) or layers[-1].in_features != Cdim:
        return None
    i, o = layers[0].in_features, layers[-1].out_features
    if not ((i == Cdim or i <= 4) and (o == Cdim or o <= 4)):
        return None
    return Cdim, (0 if i == Cdim else i), (0 if o == Cdim else o)


_BWD_MAX_LAYERS = {32: 8, 64: 8, 128: 5}      # the backward keeps every layer's slopes in registers
_FEW_TOKENS = {32: 16384, 64: 16384, 128: 12288}


class _SubChain:
    """The C x C layers of a stack whose first input and/or last output is narrow, as a stack of their own: what the
    fused launches and their backward see while gradients are enabled.  `first` / `last`: the narrow nn.Linear that
    stays a torch layer on that side (or None); the packed-weight caches live on this object."""

    num_layers = None

    def __init__(self, layers, act_mask, add_mask, act, C, first, first_act, last, act_module):
        self.__dict__["_flare_layers"] = ((layers, act_mask, add_mask, act), None)
        self.C, self.first, self.first_act, self.last, self.act_module = C, first, first_act, last, act_module


class _NarrowLinearFn(torch.autograd.Function):
    """t = x W^T + b for a Linear with a few input columns (the lift of the models' in_proj) under autocast.  Only the
    weight gradient differs from torch's own: dW = g^T x contracts over all tokens into a [C, in_dim] result, which the
    library runs as one long product with nothing to parallelise; here it is a batched product over chunks of 4096
    tokens whose partial results are summed in fp32."""

    @staticmethod
    def forward(ctx, x2, w, b, cd):
        ctx.save_for_backward(x2, w)
        ctx.has_bias = b is not None
        return torch.nn.functional.linear(x2.to(cd), w.to(cd), None if b is None else b.to(cd))

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        x2, w = ctx.saved_tensors
        T, chunk = g.shape[0], 4096
        n = T // chunk
        xc = x2.to(g.dtype)
        dw = torch.zeros(w.shape, dtype=torch.float32, device=g.device)
        if n > 0:
            dw += torch.bmm(g[:n * chunk].view(n, chunk, -1).transpose(1, 2), xc[:n * chunk].view(n, chunk, -1)).sum(0, dtype=torch.float32)
        if n * chunk < T:
            dw += (g[n * chunk:].t() @ xc[n * chunk:]).float()
        db = g.sum(0, dtype=torch.float32).to(w.dtype) if ctx.has_bias else None
        dx = (g @ w.to(g.dtype)).to(x2.dtype) if ctx.needs_input_grad[0] else None
        return dx, dw.to(w.dtype), db, None


def _narrow_ok(layer, x, cd, act_module=None):
    """True where the narrow layer (and the activation behind it) can run as one HIP pass each way: plain modules, fp32 parameters, and
    for the first layer an input that asks for no gradient."""
    w, b = layer._parameters.get("weight"), layer._parameters.get("bias")
    return (type(layer) is nn.Linear and cd in (torch.bfloat16, torch.float16) and x.is_cuda and type(x) in (torch.Tensor, nn.Parameter)
            and x.numel() > 0 and _plain_module(layer)
            and (act_module is None or (type(act_module) in (nn.GELU, nn.SiLU) and _plain_module(act_module)))
            and ("bias" in layer._parameters) and all(type(t) in (torch.Tensor, nn.Parameter) and t.dtype is torch.float32 and t.is_cuda
                                                      and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (w, b) if t is not None)
            and w is not None)


def _plain_module(m):
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or "forward" in m.__dict__
                or nn.modules.module._has_any_global_hook())


def _narrow_desc(x2, w, cd, out, act, y_dtype):
    d = _lib.FlareNarrowDesc()
    d.T, d.x_stride, d.out, d.act = x2.shape[0], x2.stride(0), int(out), act
    d.C, d.K = (w.shape[1], w.shape[0]) if out else (w.shape[0], w.shape[1])
    d.w_dtype, d.x_dtype, d.y_dtype = _DTYPES[cd], _DTYPES[x2.dtype], _DTYPES[y_dtype]
    return d


def _narrow_rows(x2):
    """Narrow rows as the launches read them: windows over a series, or one point for all tokens, are rows that share memory."""
    return x2 if x2.stride(-1) == 1 and x2.stride(0) >= x2.shape[1] else x2.clone(memory_format=torch.contiguous_format)


def _grid_rows(t):
    """Rows [T, width] as the launches read them, on the 16-byte grid and a width or more apart; others are copied (contiguous() would
    give back contiguous rows that begin off the grid)."""
    step, unit = t.stride()
    if unit == 1 and step % 4 == 0 and step >= t.shape[1] and t.data_ptr() % 16 == 0:
        return t
    return t.clone(memory_format=torch.contiguous_format)


def _narrow_backward(d, x2, w, t, dy2, dx, has_bias, dev):
    lib = _lib.load()
    parts = C.c_int32(0)
    _lib.check(lib.flare_mlp_narrow_parts(d.T, C.byref(parts)), "flare_mlp_narrow_parts")
    nb = 4 if d.out else d.C
    part = torch.empty(parts.value, w.numel() + nb, dtype=torch.float32, device=dev)
    dw, db = torch.empty_like(w), torch.empty(nb, dtype=torch.float32, device=dev)
    with _on_device(dev):
        rc = lib.flare_mlp_narrow_bwd(C.byref(d), _ptr(x2), _ptr(w), _ptr(t), _ptr(dy2), _ptr(dx), _ptr(part),
                                      part.data_ptr() + 4 * parts.value * w.numel(), _ptr(dw), _ptr(db), C.c_void_p(_stream_ptr(dev)))
    _lib.check(rc, "flare_mlp_narrow_bwd")
    return dw, (db if not d.out else db[:d.K]) if has_bias else None


class _NarrowInFn(torch.autograd.Function):
    """act(x W^T + b) of the lift in the compute type (act -1: none); x [T, in_dim] asks for no gradient."""

    @staticmethod
    def forward(ctx, x2, w, b, cd, act):
        x2 = _narrow_rows(x2)
        d = _narrow_desc(x2, w, cd, False, act, cd)
        y = torch.empty(d.T, d.C, dtype=cd, device=x2.device)
        t = torch.empty_like(y) if act >= 0 else None
        with _on_device(x2.device):
            rc = _lib.load().flare_mlp_narrow_fwd(C.byref(d), _ptr(x2), _ptr(w), _ptr(b), _ptr(t), _ptr(y), C.c_void_p(_stream_ptr(x2.device)))
        _lib.check(rc, "flare_mlp_narrow_fwd")
        ctx.cd, ctx.act, ctx.has_bias = cd, act, b is not None
        ctx.save_for_backward(x2, w, t)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        x2, w, t = ctx.saved_tensors                      # through saved-tensor hooks in any memory order
        x2 = _narrow_rows(x2)
        d = _narrow_desc(x2, w.contiguous(), ctx.cd, False, ctx.act, ctx.cd)
        dw, db = _narrow_backward(d, x2, w.contiguous(), None if t is None else _wide(t, ctx.cd), _wide(dy, ctx.cd), None, ctx.has_bias, dy.device)
        return None, dw, db, None, None


class _NarrowOutFn(torch.autograd.Function):
    """x W^T + b of the last layer in the compute type, handed out in y_dtype.  The backward of a gradient penalty on this layer's weight
    is differentiated again: then it is torch's products, with the launch's roundings."""

    @staticmethod
    def forward(ctx, x, w, b, cd, y_dtype):
        x2 = _wide(x, cd)
        d = _narrow_desc(x2, w, cd, True, -1, y_dtype)
        y = torch.empty(*x.shape[:-1], d.K, dtype=y_dtype, device=x.device)
        with _on_device(x.device):
            rc = _lib.load().flare_mlp_narrow_fwd(C.byref(d), _ptr(x2), _ptr(w), _ptr(b), None, _ptr(y), C.c_void_p(_stream_ptr(x.device)))
        _lib.check(rc, "flare_mlp_narrow_fwd")
        ctx.cd, ctx.y_dtype, ctx.has_bias, ctx.shape = cd, y_dtype, b is not None, x.shape
        ctx.save_for_backward(x, w)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        if torch.is_grad_enabled():
            with torch.autocast("cuda", enabled=False):
                g, xc, wc = (t.to(ctx.cd).float() for t in (dy.reshape(-1, dy.shape[-1]), x.reshape(-1, x.shape[-1]), w))
                return (g @ wc).to(x.dtype).view(ctx.shape), g.t() @ xc, g.sum(0) if ctx.has_bias else None, None, None
        x2, w = _wide(x, ctx.cd), w.contiguous()
        d = _narrow_desc(x2, w, ctx.cd, True, -1, ctx.y_dtype)
        dx = torch.empty_like(x2) if ctx.needs_input_grad[0] else None
        dw, db = _narrow_backward(d, x2, w, None, dy.contiguous(), dx, ctx.has_bias, dy.device)
        return None if dx is None else dx.to(x.dtype).view(ctx.shape), dw, db, None, None


def _wide(t, cd):
    """Contiguous rows [T, C] in the compute type on the 16-byte grid."""
    t = t.reshape(-1, t.shape[-1]).to(cd).contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _train_subchain(mod):
    """_SubChain of a stack with a narrow end (None for every other module); kept on the module."""
    key = _structure_key(mod)
    cached = mod.__dict__.get("_flare_subchain")
    if cached is not None and cached[1] == key:
        return cached[0]
    sub = None
    info = _layers_of(mod)
    if info is not None:
        layers, act_mask, add_mask, act = info
        io = _io_dims(mod, layers)
        if io is not None and (io[1] or io[2]):
            Cdim, in_dim, out_dim = io
            lo, hi = (1 if in_dim else 0), (len(layers) - 1 if out_dim else len(layers))
            n = hi - lo
            if n >= 1:
                keep = (1 << n) - 1
                sub = _SubChain(layers[lo:hi], (act_mask >> lo) & keep, (add_mask >> lo) & keep, act, Cdim,
                                layers[0] if in_dim else None, bool(act_mask & 1), layers[-1] if out_dim else None, mod.act)
    mod.__dict__["_flare_subchain"] = (sub, key)
    return sub


def compute_dtype(x, mod):
    """The 16-bit type the fused kernels may run this module in, or None (then torch runs it).  With gradients
    enabled the chain of C x C layers and the expanding two-layer MLP qualify (the shapes flare_mlp_bwd and
    flare_mlp_expand_bwd differentiate), and a stack with a narrow end for the chain between its narrow layers."""
    if x.device.type != "cuda":
        return None
    # what depends on the module's structure and the row width only is decided once per (structure, width, grad mode)
    grad = torch.is_grad_enabled()
    key = (_structure_key(mod), x.shape[-1], grad)
    cached = mod.__dict__.get("_flare_shape_ok")
    if cached is None or cached[0] != key:
        cached = (key, _shape_ok(x.shape[-1], mod, grad))
        mod.__dict__["_flare_shape_ok"] = cached
    if not cached[1]:
        return None
    layers = _layers_of(mod)[0]
    if x.dtype not in (torch.float32, torch.bfloat16, torch.float16) or x.stride(-1) != 1:
        return None
    ac = _autocast_dtype(x)
    if ac in (torch.bfloat16, torch.float16):
        return ac
    wd = layers[0].weight.dtype
    if ac is None and wd in (torch.bfloat16, torch.float16) and all(l.weight.dtype == wd for l in layers):
        return wd
    return None


def _shape_ok(width, mod, grad):
    info = _layers_of(mod)
    if info is None:
        return False
    layers = info[0]
    if len(layers) > 16:
        return False
    if grad:
        sub = _train_subchain(mod)
        if sub is not None:                 # narrow first input / last output: the C x C layers between them
            n = len(_layers_of(sub)[0])
            if sub.C not in _SUPPORTED_C or n > _BWD_MAX_LAYERS[sub.C] or width != layers[0].in_features:
                return False
        else:
            if width not in _SUPPORTED_C:
                return False
            if not _expand_factor(mod, width):
                if len(layers) > _BWD_MAX_LAYERS[width] or any(l.in_features != width or l.out_features != width for l in layers):
                    return False
    io = _io_dims(mod, layers)
    if io is not None and (io[1] or io[2]):
        if io[0] not in _SUPPORTED_C or width != layers[0].in_features:
            return False
    else:
        if width not in _SUPPORTED_C:
            return False
        if not _expand_factor(mod, width) and any(l.in_features != width or l.out_features != width for l in layers):
            return False
    return True


def _readable(*ts):
    """The packing launch reads these parameters where they lie (a tensor subclass may keep its values elsewhere)."""
    return all(t is None or (type(t) in (torch.Tensor, nn.Parameter) and t.is_cuda and t.dtype in _DTYPES
                             and t.stride(-1) == 1 and (t.dim() == 1 or t.stride(0) >= t.shape[1])) for t in ts)


def _pack_launch(Cdim, cd, tiles, dev, images, tiled=False, latents=None):
    """One flare_mlp_pack launch.  tiles: (weight, element offset of the tile, row stride, rows, bias or None, element offset)
    each; returns (w [L,C,C], b [L,C], image of w, image of its transposes), the images None unless asked for.  tiled: w and the
    last result in the few-token kernels' operand order, no image of w.  latents: (values, 16-bit result [..., columns]) converted and
    zero-padded on the way."""
    lib = _lib.load()
    L = len(tiles)
    d = _lib.FlareMlpPackDesc()
    d.L, d.C, d.w_dtype = L, Cdim, _DTYPES[cd]
    for l, (w, off, ld, rows, b, boff) in enumerate(tiles):
        d.src[l], d.ld[l], d.rows[l], d.src_dtype[l] = w.data_ptr() + off * w.element_size(), ld, rows, _DTYPES[w.dtype]
        if b is not None:
            d.bsrc[l], d.b_dtype[l] = b.data_ptr() + boff * b.element_size(), _DTYPES[b.dtype]
    d.tiled = int(tiled)
    ws = torch.empty(1 if not images else 2 if tiled else 3, L, Cdim, Cdim, dtype=cd, device=dev)
    bias = torch.empty(L, Cdim, dtype=torch.float32, device=dev)
    with _on_device(dev):
        img = ws[1] if images and not tiled else None
        img_t = ws[-1] if images else None
        src, out = latents or (None, None)
        n, cols, cols_out, dt = (0, 0, 0, 0) if latents is None else (src.numel() // src.shape[-1], src.shape[-1], out.shape[-1], _DTYPES[src.dtype])
        rc = lib.flare_mlp_pack_rows(C.byref(d), _ptr(ws), _ptr(img), _ptr(img_t), _ptr(bias), _ptr(src), n, cols, cols_out, dt, _ptr(out),
                                     C.c_void_p(_stream_ptr(dev)))
    _lib.check(rc, "flare_mlp_pack_rows")
    return ws[0], bias, img, img_t


def _chain_tiles(layers):
    """Tiles of a stack of Linears at most C x C, or None where the launch cannot read them."""
    tiles = []
    for l in layers:
        p = l._parameters                      # as in _param_key: a model's first forward comes here for every layer
        w, b = (p["weight"], p["bias"]) if "weight" in p and "bias" in p else (l.weight, l.bias)
        if not _readable(w, b):
            return None
        tiles.append((w, 0, w.stride(0), l.out_features, b, 0))
    return tiles


def _expand_tiles(f1, f2, E, Cdim):
    if not _readable(f1.weight, f1.bias, f2.weight, f2.bias):
        return None
    w1, w2, tiles = f1.weight, f2.weight, []
    for j in range(E):
        tiles.append((w1, j * Cdim * w1.stride(0), w1.stride(0), Cdim, f1.bias, j * Cdim))
        tiles.append((w2, j * Cdim, w2.stride(0), Cdim, f2.bias if j == 0 else None, 0))
    return tiles


def _few(T, Cdim, L):
    """Rows of the norm's partial sums the few-token backward writes for such a launch, 0 where the other kernels serve it:
    what flare_mlp_few answers, without a call into the library (every fused call asks)."""
    return (T + 15) // 16 if 0 < T <= _FEW_TOKENS.get(Cdim, 0) and L <= _BWD_MAX_LAYERS[Cdim] else 0


def _param_key(layers):
    """What packed copies of these layers' parameters depend on: an in-place change moves a version, another tensor an address (see
    _Key).  Read from the layers' own tables (see _structure_key); a parametrised weight is another tensor at every access, so copies of it
    serve one call."""
    key = []
    for l in layers:
        p = l._parameters
        if "weight" not in p or "bias" not in p:
            key.append((object(),))
            continue
        w, b = p["weight"], p["bias"]
        key.append((w.data_ptr(), w._version) if b is None else (w.data_ptr(), w._version, b.data_ptr(), b._version))
    return tuple(key)


_KEPT = frozenset(("_flare_plans", "_q_cache", "_flare_subchain", "_flare_packed", "_flare_packed_train", "_flare_packed_few"))      # see drop_operands


class DropsOperands:
    """For modules: to(), cpu(), half() and their like drop what is kept of parameters that they replace.  Where they leave all of them in
    place the packed copies stay: a graph that the caller has recorded may read them."""

    def _apply(self, fn, recurse=True):
        # its own and, for plain layers among them, its children's: every module that keeps more is of this kind itself
        kept = [m for m in (self, *self._modules.values()) if m is not None and not _KEPT.isdisjoint(m.__dict__)]
        if not kept:
            return super()._apply(fn, recurse)
        before = [(t.data_ptr(), t.dtype) for t in self.parameters()]
        out = super()._apply(fn, recurse)
        if before != [(t.data_ptr(), t.dtype) for t in self.parameters()]:
            for m in kept:
                drop_operands(m)
        return out


class _Key(tuple):
    """The key of something kept.  held: the memory whose addresses it names (hold()), so that no other tensor gets one of them while
    it is compared.  A copy of a module, and one read back from a file, holds nothing: there the key fits no tensor."""

    def __deepcopy__(self, memo):
        return ()

    def __reduce__(self):
        return tuple, ()


def hold(t):
    """Something that keeps t's memory from being given to others, also when t is given other memory (a storage, of a plain tensor: a
    sixth of a detach(), and a model's first forward holds hundreds)."""
    return t.untyped_storage() if type(t) in (torch.Tensor, nn.Parameter) else t.detach()


def _kept(key, layers):
    """A cache's first entry for key, which names these layers' parameters."""
    kept = _Key(key)
    kept.held = [t.untyped_storage() if type(t) is nn.Parameter else hold(t) for l in layers for t in l._parameters.values() if t is not None]
    return kept


def drop_operands(mod):
    """Forget the packed weights kept for mod, for the chain between its narrow ends (that chain's copies live on an object that
    is no submodule, and a walk over module.modules() alone passes them by), a block's plans, which hold copies of their own, and the
    latents' cast copy."""
    mod.__dict__.pop("_flare_plans", None)
    mod.__dict__.pop("_q_cache", None)
    sub = mod.__dict__.get("_flare_subchain")
    for m in (mod, None if sub is None else sub[0]):
        if m is not None:
            for name in ("_flare_packed", "_flare_packed_train", "_flare_packed_few"):
                m.__dict__.pop(name, None)


def _packed_few(mod, layers, cd, train):
    """(tiled w, fp32 biases, tiled transposes or None) of a chain for the few-token launches, cached on the module; None where
    the packing launch cannot read the parameters.  A pair passes the layers of both stacks and the first stack's module."""
    key = (cd, _param_key(layers))
    cache = mod.__dict__.get("_flare_packed_few")
    if cache is not None and cache[0] == key and (cache[3] is not None or not train):
        return cache[1:]
    tiles = _chain_tiles(layers)
    if tiles is None:
        return None
    w, b, _, wt = _pack_launch(layers[0].in_features, cd, tiles, layers[0].weight.device, train, tiled=True)
    mod.__dict__["_flare_packed_few"] = (_kept(key, layers), w, b, wt)
    return w, b, wt


def _packed(mod, layers, cd):
    """[L,C,C] weights in the compute dtype and [L,C] fp32 biases, cached on the module."""
    key = (cd, _param_key(layers))
    cache = getattr(mod, "_flare_packed", None)
    if cache is not None and cache[0] == key:
        return cache[1], cache[2]
    tiles = _chain_tiles(layers)
    if tiles is not None:
        w, b, _, _ = _pack_launch(layers[0].in_features, cd, tiles, layers[0].weight.device, False)
        mod._flare_packed = (_kept(key, layers), w, b)
        return w, b
    w = torch.stack([l.weight.detach() for l in layers]).to(cd).contiguous()
    Cdim = w.shape[-1]
    b = torch.stack([l.bias.detach().float() if l.bias is not None else w.new_zeros(Cdim, dtype=torch.float32) for l in layers]).contiguous()
    mod._flare_packed = (_kept(key, layers), w, b)
    return w, b


def _packed_expand(mod, E, cd):
    """Tiles W1[0:C], W2[:,0:C], W1[C:2C], W2[:,C:2C], ... as [2E,C,C] and bias rows b1[0:C], b2, b1[C:2C], 0, ...
    (the layout FLARE_MLP_EXPAND asks for), cached on the module."""
    f1, f2 = mod.fc1, mod.fc2
    key = ("expand", cd, _param_key((f1, f2)))
    cache = getattr(mod, "_flare_packed", None)
    if cache is not None and cache[0] == key:
        return cache[1], cache[2]
    Cdim = f1.in_features
    tiles = _expand_tiles(f1, f2, E, Cdim)
    if tiles is not None:
        w, b, _, _ = _pack_launch(Cdim, cd, tiles, f1.weight.device, False)
        mod._flare_packed = (_kept(key, (f1, f2)), w, b)
        return w, b
    w1 = f1.weight.detach().to(cd).view(E, Cdim, Cdim)                       # [j][hidden row in chunk][in]
    w2 = f2.weight.detach().to(cd).view(Cdim, E, Cdim).permute(1, 0, 2)      # [j][out][hidden col in chunk]
    w = torch.stack([w1, w2], dim=1).reshape(2 * E, Cdim, Cdim).contiguous()
    b = torch.zeros(2 * E, Cdim, dtype=torch.float32, device=w.device)
    if f1.bias is not None:
        b[0::2] = f1.bias.detach().float().view(E, Cdim)
    if f2.bias is not None:
        b[1] = f2.bias.detach().float()
    mod._flare_packed = (_kept(key, (f1, f2)), w, b)
    return w, b


def _packed_io(mod, layers, cd, Cdim, in_dim, out_dim):
    """Tiles of a stack with a narrow first and/or last layer: (w [L,C,C], b [L,C], w_in [C,4] fp32, b_in [C]),
    the narrow last layer zero-padded to C rows; cached on the module."""
    key = ("io", cd, _param_key(layers))
    cache = getattr(mod, "_flare_packed", None)
    if cache is not None and cache[0] == key:
        return cache[1:]
    dev = layers[0].weight.device
    tiles = layers[1:] if in_dim else layers
    packed = _chain_tiles(tiles)
    if packed is not None:
        w, b, _, _ = _pack_launch(Cdim, cd, packed, dev, False)
    else:
        w = torch.zeros(len(tiles), Cdim, Cdim, dtype=cd, device=dev)
        b = torch.zeros(len(tiles), Cdim, dtype=torch.float32, device=dev)
        for i, l in enumerate(tiles):
            w[i, :l.out_features] = l.weight.detach().to(cd)
            if l.bias is not None:
                b[i, :l.out_features] = l.bias.detach().float()
    w_in = b_in = None
    if in_dim:
        w_in = torch.zeros(Cdim, 4, dtype=torch.float32, device=dev)
        w_in[:, :in_dim] = layers[0].weight.detach().float()
        b_in = (layers[0].bias.detach().float().contiguous() if layers[0].bias is not None
                else torch.zeros(Cdim, dtype=torch.float32, device=dev))
    mod._flare_packed = (_kept(key, layers), w, b, w_in, b_in)
    return w, b, w_in, b_in


def _fused_mlp_io(x, mod, cd, io, info, norm, out_dtype):
    lib = _lib.load()
    layers, act_mask, add_mask, act = info
    Cdim, in_dim, out_dim = io
    w, b, w_in, b_in = _packed_io(mod, layers, cd, Cdim, in_dim, out_dim)
    in_act = act_mask & 1
    if in_dim:                       # the first layer is not one of the tiles
        act_mask >>= 1
        add_mask >>= 1
    xw = x.shape[-1]
    x2 = x.reshape(-1, xw)
    x2 = _narrow_rows(x2) if in_dim else _grid_rows(x2)
    out_dtype = x.dtype if out_dtype is None else out_dtype
    yw = out_dim if out_dim else Cdim
    y = torch.empty(*x.shape[:-1], yw, dtype=out_dtype, device=x.device)
    d = _lib.FlareMlpDesc()
    d.T, d.C, d.L = x2.shape[0], Cdim, w.shape[0]
    d.w_dtype, d.x_dtype, d.y_dtype = _dtype_code(w), _dtype_code(x2), _dtype_code(y)
    d.act, d.act_mask, d.add_mask = act, act_mask, add_mask
    d.x_stride, d.y_stride = x2.stride(0), yw
    gamma, beta = _norm_args(d, norm, x, Cdim)
    with _on_device(x.device):
        rc = lib.flare_mlp_io_fwd(C.byref(d), in_dim, in_act, _ptr(w_in), _ptr(b_in), out_dim, _ptr(x2), _ptr(w), _ptr(b),
                                  _ptr(gamma), _ptr(beta), None, _ptr(y), C.c_void_p(_stream_ptr(x.device)))
    _lib.check(rc, "flare_mlp_io_fwd")
    return y


def _vec32(p):
    """A parameter vector as the launches read it: itself where it already is contiguous fp32 on the 16-byte grid."""
    if p.dtype is torch.float32 and p.is_contiguous() and type(p) in (torch.Tensor, nn.Parameter) and p.data_ptr() % 16 == 0:
        return p
    v = p.detach().float().contiguous()
    return v if v.data_ptr() % 16 == 0 else v.clone()


def _norm_args(d, norm, x, Cdim, vectors=None):
    """Fill the descriptor's norm fields; returns (gamma, beta) fp32 tensors or None.  vectors: (weight, bias) in place of the norm's own."""
    gamma = beta = None
    if norm is not None and not isinstance(norm, nn.Identity):
        if isinstance(norm, nn.LayerNorm):
            d.norm, d.eps = 1, float(norm.eps)
            bias = norm.bias if vectors is None else vectors[1]
            beta = None if bias is None else _vec32(bias)
        elif isinstance(norm, nn.RMSNorm):
            d.norm = 2
            d.eps = float(norm.eps) if norm.eps is not None else float(torch.finfo(x.dtype).eps)
        else:
            raise TypeError(f"unsupported norm {type(norm).__name__}")
        weight = norm.weight if vectors is None else vectors[0]
        gamma = _vec32(weight) if weight is not None else torch.ones(Cdim, dtype=torch.float32, device=x.device)
    return gamma, beta


def fused_mlp(x, mod, cd, norm=None, res=None, out_dtype=None, x_head=0, y_head=0):
    """y = res + mod(norm(x)) in one HIP launch.  x: [..., C]; mod: ResidualMLP or nn.Linear; cd: the
    dtype from compute_dtype(); norm: nn.LayerNorm / nn.RMSNorm / None; res: [..., C] or None.
    x_head / y_head (4 or 8): x is / y comes back head-padded, [..., (C / head) * 16] with every head's channels
    followed by zeros up to 16 columns -- the layout the mixer reads and writes for head dims below 16.
    With gradients enabled the call is differentiable (chain of C x C layers only, see compute_dtype)."""
    if torch.is_grad_enabled():
        if x_head or y_head:
            raise ValueError("head-padded rows have no backward: call under torch.no_grad()")
        sub = _train_subchain(mod)
        if sub is not None:
            # narrow ends: those layers run as torch layers (under the caller's autocast), the chain between them fused
            out_dtype = x.dtype if out_dtype is None else out_dtype
            h, hn = x, norm
            if sub.first is not None:
                if hn is not None and not isinstance(hn, nn.Identity):
                    h, hn = hn(h), None
                h2 = h.reshape(-1, h.shape[-1])
                if not h.requires_grad and _narrow_ok(sub.first, h, cd, sub.act_module if sub.first_act else None):
                    act = _layers_of(sub)[3] if sub.first_act else -1
                    h = _NarrowInFn.apply(h2, sub.first.weight, sub.first.bias, cd, act).view(*h.shape[:-1], -1)
                else:
                    h = _NarrowLinearFn.apply(h2, sub.first.weight, sub.first.bias, cd).view(*h.shape[:-1], -1)
                    if sub.first_act:
                        h = sub.act_module(h)
            y = _fused_mlp_train(h, sub, cd, hn, None, cd if sub.last is not None else out_dtype)
            if sub.last is not None:
                if out_dtype in _DTYPES and _narrow_ok(sub.last, y, cd):
                    y = _NarrowOutFn.apply(y, sub.last.weight, sub.last.bias, cd, out_dtype)
                else:
                    y = sub.last(y).to(out_dtype)
            return y if res is None else res + y
        return _fused_mlp_train(x, mod, cd, norm, res, out_dtype)
    return _fused_mlp_fwd(x, mod, cd, norm, res, out_dtype, x_head, y_head)


def _pair_info(x, mod_a, mod_b, cd):
    """(layers of both, act_mask, add_mask, act) where one few-token launch takes both stacks, else None: plain chains of
    C x C layers, alike in length, masks and activation, and few enough tokens."""
    Cdim = x.shape[-1]
    if not 0 < x.numel() // Cdim <= _FEW_TOKENS.get(Cdim, 0):      # most calls end here: nothing else is looked at for them
        return None
    infos = [_layers_of(m) for m in (mod_a, mod_b)]
    if infos[0] is None or infos[1] is None or infos[0][1:] != infos[1][1:] or len(infos[0][0]) != len(infos[1][0]):
        return None
    layers = infos[0][0] + infos[1][0]
    if len(layers) > _lib.MLP_PACK_MAX or any(l.in_features != Cdim or l.out_features != Cdim for l in layers):
        return None
    if not _few(x.numel() // Cdim, Cdim, len(infos[0][0])):
        return None
    return (layers, *infos[0][1:])


def narrow_train_ok(x, mod_a, mod_b, out):
    """True where a training step may keep narrow heads padded between the projections, the mixer and the output projection: the
    few-token launches differentiate head-padded rows (x: the rows the projections read; out: a Linear of their width)."""
    info = _pair_info(x, mod_a, mod_b, None)
    return (info is not None and isinstance(out, nn.Linear) and _train_subchain(mod_a) is None and _train_subchain(mod_b) is None
            and out.in_features == out.out_features == x.shape[-1] and _chain_tiles(info[0] + [out]) is not None)


def _pair_packs(x, mod_a, mod_b):
    info = _pair_info(x, mod_a, mod_b, None)
    return info is not None and _chain_tiles(info[0]) is not None


def prepack(x, cd, *stacks, latents=None):
    """The packed operands of several stacks that the few-token launches of one training step will ask for (a tuple of modules shares
    a packing: a pair), from one packing launch instead of one each.  Does nothing where they are not all plain chains at few
    tokens, or where fewer than two of them have to be packed again.  latents: see _pack_launch; True if they have been converted."""
    Cdim = x.shape[-1]
    if not 0 < x.numel() // Cdim <= _FEW_TOKENS.get(Cdim, 0):
        return
    stale, tiles, at = [], [], 0
    for mods in stacks:
        layers = []
        for m in mods:
            info = _layers_of(m)
            if (info is None or len(info[0]) > _BWD_MAX_LAYERS[Cdim] or _train_subchain(m) is not None
                    or any(l.in_features != Cdim or l.out_features != Cdim for l in info[0])):
                return
            layers += info[0]
        if len(mods) == 2 and _pair_info(x, *mods, cd) is None:
            return
        key = (cd, _param_key(layers))
        cache = mods[0].__dict__.get("_flare_packed_few")
        if cache is not None and cache[0] == key and cache[3] is not None:
            continue
        t = _chain_tiles(layers)
        if t is None:
            return
        stale.append((mods[0], _kept(key, layers), at, at + len(t)))
        tiles += t
        at += len(t)
    if len(stale) < 2 or at > _lib.MLP_PACK_MAX:
        return
    w, b, _, wt = _pack_launch(Cdim, cd, tiles, x.device, True, tiled=True, latents=latents)
    for mod, key, lo, hi in stale:
        mod.__dict__["_flare_packed_few"] = (key, w[lo:hi], b[lo:hi], wt[lo:hi])
    return True


def project_padded(y, out, cd, head, res, out_dtype):
    """[res +] out(y) for rows y of padded heads, differentiable where narrow_train_ok() says so."""
    if torch.is_grad_enabled():
        return _fused_mlp_train(y, out, cd, None, res, out_dtype, head)
    return fused_mlp(y, out, cd, res=res, out_dtype=out_dtype, x_head=head)


def fused_mlp_pair(x, mod_a, mod_b, cd, norm=None, out_dtype=None, y_head=0, with_res=False):
    """(mod_a(norm(x)), mod_b(norm(x))) as fused_mlp computes them, for two stacks that read the same rows through the
    same norm (a block's k and v projections).  With gradients enabled and both stacks plain chains of C x C layers the
    pair is one autograd node whose backward sums the two gradients of x inside the second launch (few tokens: one backward
    launch for both stacks).  y_head: as fused_mlp's, with gradients enabled where narrow_train_ok() says so.
    with_res: a third result, x as the block's residual is to read it: where one launch is the pair's backward, that path's gradient
    is added there, and not by a launch over three [T, C] arrays."""
    if torch.is_grad_enabled() and all(_train_subchain(m) is None and not _expand_factor(m, x.shape[-1]) for m in (mod_a, mod_b)):
        has_norm = norm is not None and not isinstance(norm, nn.Identity)
        gamma = getattr(norm, "weight", None) if has_norm else None
        beta = getattr(norm, "bias", None) if has_norm else None
        wb = []
        for m in (mod_a, mod_b):
            layers = _layers_of(m)[0]
            wb += [l.weight for l in layers] + [l.bias for l in layers]
        through = with_res and x.requires_grad and type(x) is torch.Tensor and _pair_packs(x, mod_a, mod_b)
        out = _FusedPairFn.apply(mod_a, mod_b, cd, norm if has_norm else None, (out_dtype, y_head, through), x, gamma, beta, *wb)
        return out if through or not with_res else (*out, x)
    out = (fused_mlp(x, mod_a, cd, norm=norm, out_dtype=out_dtype, y_head=y_head),
           fused_mlp(x, mod_b, cd, norm=norm, out_dtype=out_dtype, y_head=y_head))
    return (*out, x) if with_res else out


def _forward_plan(mod):
    """(_layers_of, _io_dims where an end is narrow else None, width, _expand_factor), kept like _layers_of."""
    key = _structure_key(mod)
    cached = mod.__dict__.get("_flare_fwd_plan")
    if cached is None or cached[1] != key:
        info = _layers_of(mod)
        io = _io_dims(mod, info[0])
        Cdim = info[0][0].in_features
        cached = ((info, io if io is not None and (io[1] or io[2]) else None, Cdim, _expand_factor(mod, Cdim)), key)
        mod.__dict__["_flare_fwd_plan"] = cached
    return cached[0]


def _fused_mlp_fwd(x, mod, cd, norm=None, res=None, out_dtype=None, x_head=0, y_head=0, train=False, operands=None, pair=None):
    """operands: the packed weights to read in place of the module's.  pair: a list that the two chains of a few-token pair pass through
    (operands: their halves of one packing): the first one's launch is left to the second."""
    lib = _lib.load()
    info, io, Cdim, E = _forward_plan(mod)
    layers, act_mask, add_mask, act = info
    if io is not None:
        y = _fused_mlp_io(x, mod, cd, io, info, norm, out_dtype)
        return y if res is None else res + y
    if x.shape[-1] != (Cdim // x_head * 16 if x_head else Cdim):
        raise ValueError(f"x rows are {x.shape[-1]} wide, expected {Cdim // x_head * 16 if x_head else Cdim}")
    few = not E and bool(_few(x.numel() // x.shape[-1], Cdim, len(layers)))
    if operands is None and few:
        operands = _packed_few(mod, layers, cd, train)
    few = few and operands is not None and len(operands) < 4
    if E and (x_head or y_head):
        raise ValueError("head-padded rows are not available for the expanding two-layer MLP")
    if operands is not None:
        w, b = operands[:2]
    elif E:
        w, b = _packed_train_expand(mod, E, cd)[:2] if train else _packed_expand(mod, E, cd)
    else:
        w, b = _packed_train(mod, layers, cd)[:2] if train else _packed(mod, layers, cd)
    if E:
        act_mask, add_mask = 1, 0
    x2 = x.reshape(-1, x.shape[-1])
    x2 = _grid_rows(x2)
    out_dtype = x.dtype if out_dtype is None else out_dtype
    ywidth = Cdim // y_head * 16 if y_head else Cdim
    y = torch.empty(*x.shape[:-1], ywidth, dtype=out_dtype, device=x.device)
    d = _lib.FlareMlpDesc()
    d.T, d.C, d.L = x2.shape[0], Cdim, w.shape[0]
    d.flags = (_lib.MLP_EXPAND if E else _lib.MLP_W_TILED if few else 0) | ((x_head // 4) << 8) | ((y_head // 4) << 12)
    d.w_dtype, d.x_dtype, d.y_dtype = _dtype_code(w), _dtype_code(x2), _dtype_code(y)
    d.act, d.act_mask, d.add_mask = act, act_mask, add_mask
    d.x_stride, d.y_stride = x2.stride(0), ywidth
    gamma, beta = _norm_args(d, norm, x, Cdim)
    r2 = None
    if res is not None:
        r2 = res.reshape(-1, Cdim)
        r2 = _grid_rows(r2)
        d.res_dtype, d.res_stride = _dtype_code(r2), r2.stride(0)
    if pair is not None:
        pair.append((w, b, y))
        if len(pair) == 2:
            (w, b, ya), _ = pair
            with _on_device(x.device):
                rc = lib.flare_mlp_few_pair_fwd(C.byref(d), _ptr(x2), _ptr(w), _ptr(b), _ptr(gamma), _ptr(beta), _ptr(ya), _ptr(y),
                                                C.c_void_p(_stream_ptr(x.device)))
            _lib.check(rc, "flare_mlp_few_pair_fwd")
        return y
    with _on_device(x.device):
        rc = lib.flare_mlp_fwd(C.byref(d), _ptr(x2), _ptr(w), _ptr(b), _ptr(gamma), _ptr(beta), _ptr(r2), _ptr(y),
                               C.c_void_p(_stream_ptr(x.device)))
    _lib.check(rc, "flare_mlp_fwd")
    return y


def _train_operands(x, mod, cd):
    """What a stack's launches read in a training step, forward and backward: the result of _packed_few (three), or of _packed_train or
    _packed_train_expand (four)."""
    info, _, Cdim, E = _forward_plan(mod)
    if E:
        return _packed_train_expand(mod, E, cd)
    packed = _packed_few(mod, info[0], cd, True) if _few(x.numel() // x.shape[-1], Cdim, len(info[0])) else None
    return _packed_train(mod, info[0], cd) if packed is None else packed


def _tail_descs(y2, out, x, mlp, cd, norm, head, vectors=None):
    """(Linear, chain) descriptors of a block's end, the norm's vectors."""
    Cdim, (layers, act_mask, add_mask, act) = out.in_features, _layers_of(mlp)
    f, s = _lib.FlareMlpDesc(), _lib.FlareMlpDesc()
    f.T = s.T = y2.shape[0]
    f.C = s.C = Cdim
    f.L, s.L = 1, len(layers)
    f.flags = (head // 4) << 8
    f.w_dtype = s.w_dtype = f.x_dtype = _DTYPES[cd]
    f.y_dtype = f.res_dtype = s.x_dtype = s.y_dtype = s.res_dtype = _dtype_code(x)
    s.act, s.act_mask, s.add_mask = act, act_mask, add_mask
    f.x_stride = y2.shape[1]
    f.y_stride = f.res_stride = s.x_stride = s.y_stride = s.res_stride = Cdim
    return (f, s, *_norm_args(s, norm, x, Cdim, vectors))


def tail_operands(out, mlp, cd):
    """What both launches of a block's end read: the packed weights of out and of mlp."""
    return _packed_few(out, [out], cd, True), _packed_few(mlp, _layers_of(mlp)[0], cd, True)


def tail_forward(y2, out, x, mlp, cd, norm, head, operands=None):
    """x1 = x + out(y2), x1 + mlp(norm(x1)) in one launch (few tokens; contiguous rows, y2 in the compute type with heads of `head`
    channels padded): (x1, result).  operands: tail_operands() of these modules."""
    y2 = y2.reshape(-1, y2.shape[-1])
    f, s, gamma, beta = _tail_descs(y2, out, x, mlp, cd, norm, head)
    f.flags, s.flags = f.flags | _lib.MLP_W_TILED, _lib.MLP_W_TILED
    (w1, b1, _), (w2, b2, _) = tail_operands(out, mlp, cd) if operands is None else operands
    x1, y = torch.empty_like(x), torch.empty_like(x)
    with _on_device(x.device):
        rc = _lib.load().flare_mlp_few_tail_fwd(C.byref(f), C.byref(s), _ptr(y2), _ptr(x), _ptr(w1), _ptr(b1), _ptr(w2), _ptr(b2), _ptr(gamma),
                                                _ptr(beta), _ptr(x1), _ptr(y), C.c_void_p(_stream_ptr(x.device)))
    _lib.check(rc, "flare_mlp_few_tail_fwd")
    return x1, y


def tail_backward(y2, out, x1, mlp, cd, norm, head, dy, a_in, g_out, operands=None, vectors=None):
    """Backward of tail_forward in one launch: (dx1 [T,C], dy2, the norm's partial rows); a_in, g_out take the rows for the weight
    gradients of out and of mlp's layers, in that order.  operands, vectors: what the forward read, of the stacks and of the norm."""
    Cdim = out.in_features
    x2, y2, dy = x1.reshape(-1, Cdim), y2.reshape(-1, y2.shape[-1]), _rows2d(dy, Cdim)
    f, s, gamma, beta = _tail_descs(y2, out, x1, mlp, cd, norm, head, vectors)
    s.y_dtype, s.y_stride = _dtype_code(dy), dy.stride(0)
    (_, _, wt1), (w2, b2, wt2) = tail_operands(out, mlp, cd) if operands is None else operands
    dx1, dy2 = torch.empty_like(x2), torch.empty_like(y2)
    gb = torch.empty(_few(x2.shape[0], Cdim, s.L), 2, Cdim, dtype=torch.float32, device=x1.device)
    with _on_device(x1.device):
        rc = _lib.load().flare_mlp_few_tail_bwd(C.byref(f), C.byref(s), _ptr(x2), _ptr(dy), _ptr(w2), _ptr(wt2), _ptr(b2), _ptr(gamma), _ptr(beta),
                                                _ptr(dx1), _ptr(a_in[1:]), _ptr(g_out[1:]), _ptr(gb), _ptr(y2), _ptr(wt1), _ptr(dy2),
                                                _ptr(a_in), _ptr(g_out), C.c_void_p(_stream_ptr(x1.device)))
    _lib.check(rc, "flare_mlp_few_tail_bwd")
    return dx1, dy2, gb


# --------------------------------------------------------------------------------------
# training: forward launch + flare_mlp_bwd
# --------------------------------------------------------------------------------------
_IMG_INDEX = {}


def _image_index(Cdim, device):
    """For every 16-bit position of a weight tile's LDS image, the row-major element that sits there (the inverse of
    the formula in include/flare_hip.h): element (row, col) of the tile is the A operand of output row `row`, and
    the kernels read 8 consecutive k-slots per lane."""
    key = (Cdim, str(device))
    idx = _IMG_INDEX.get(key)
    if idx is None:
        sws = {128: 0, 64: 1, 32: 2}[Cdim]
        row = torch.arange(Cdim).view(-1, 1).expand(Cdim, Cdim)
        col = torch.arange(Cdim).view(1, -1).expand(Cdim, Cdim)
        ch, j = col // 8, col % 8
        chunk = 4 * (ch // 4) + 2 * (ch % 2) + j // 4
        pos = row * Cdim + 8 * (chunk ^ ((row % 16) >> sws)) + 4 * ((ch % 4) // 2) + j % 4
        idx = torch.empty(Cdim * Cdim, dtype=torch.long)
        idx[pos.reshape(-1)] = torch.arange(Cdim * Cdim)
        idx = _IMG_INDEX[key] = idx.to(device)
    return idx


def mlp_weight_image(w):
    """[L,C,C] weights ([out][in] per tile) -> the LDS images flare_mlp_bwd loads straight into its weight slots."""
    L, Cdim, _ = w.shape
    return w.reshape(L, Cdim * Cdim)[:, _image_index(Cdim, w.device)].contiguous()


_IMG_INDEX2 = {}


def mlp_weight_images(w):
    """(image of w, image of its transposes) as one gather: the transposed tile's element (row, col) is w[col][row], so
    its image reads w through the same index with row and column swapped.  A training step packs after every
    optimizer update, and on small meshes each saved launch counts."""
    L, Cdim, _ = w.shape
    key = (Cdim, L, str(w.device))
    ix = _IMG_INDEX2.get(key)
    if ix is None:
        idx = _image_index(Cdim, w.device)
        both = torch.stack([idx, (idx % Cdim) * Cdim + idx // Cdim])                     # [2, C*C]
        ix = _IMG_INDEX2[key] = (torch.arange(L, device=w.device).view(1, L, 1), both.view(2, 1, Cdim * Cdim))
    imgs = w.reshape(L, Cdim * Cdim)[ix[0], ix[1]]                                          # [2, L, C*C], contiguous
    return imgs[0], imgs[1]


def _packed_train(mod, layers, cd):
    """(w [L,C,C] for the forward launch, images of the weights and of their transposes for the backward, fp32 biases
    [L,C]), cached on the module until a parameter changes."""
    key = ("train", cd, _param_key(layers))
    cache = mod.__dict__.get("_flare_packed_train")
    if cache is not None and cache[0] == key:
        return cache[1:]
    tiles = _chain_tiles(layers)
    if tiles is not None:
        w, b, w_img, wt_img = _pack_launch(layers[0].in_features, cd, tiles, layers[0].weight.device, True)
    else:
        w, b = _packed(mod, layers, cd)
        w_img, wt_img = mlp_weight_images(w)
    mod.__dict__["_flare_packed_train"] = (_kept(key, layers), w, b, w_img, wt_img)
    return w, b, w_img, wt_img


def _packed_train_expand(mod, E, cd):
    """The same for the expanding two-layer MLP: its 2 E tiles (see _packed_expand) and their transposes as images."""
    f1, f2 = mod.fc1, mod.fc2
    key = ("train-expand", cd, _param_key((f1, f2)))
    cache = mod.__dict__.get("_flare_packed_train")
    if cache is not None and cache[0] == key:
        return cache[1:]
    tiles = _expand_tiles(f1, f2, E, f1.in_features)
    if tiles is not None:
        w, b, w_img, wt_img = _pack_launch(f1.in_features, cd, tiles, f1.weight.device, True)
    else:
        w, b = _packed_expand(mod, E, cd)
        w_img, wt_img = mlp_weight_images(w)
    mod.__dict__["_flare_packed_train"] = (_kept(key, (f1, f2)), w, b, w_img, wt_img)
    return w, b, w_img, wt_img


def _weight_grads(d, g_out, a_in, want_bias, L=None, gb=None, gsum=None, gb2=None, gsum2=None, latents=None, dq=None):
    """dW [L, C(out), C(in)] and db [L, C] (or None) in fp32 from the rows the backward launch left: one pass of
    flare_mlp_wgrad over both row arrays, partial results per token range summed in a fixed order.  g_out, a_in:
    [L,T,C], or [T,C] for an array all L layers share.  gb, gsum: the norm's partial rows [rows,2,C], summed into gsum [2,C] by
    the launch that sums the others; gb2, gsum2: another norm's; latents, dq: what _mixer_hip_grad left of the latents' gradient,
    summed into dq [H,M,columns]."""
    lib = _lib.load()
    T, Cdim = g_out.shape[-2:]
    L = (g_out.shape[0] if g_out.dim() == 3 else a_in.shape[0]) if L is None else L
    d2 = _lib.FlareMlpDesc()
    d2.T, d2.C, d2.L, d2.w_dtype = T, Cdim, L, d.w_dtype
    d = d2
    parts = C.c_int32(0)
    _lib.check(lib.flare_mlp_wgrad_partials(C.byref(d), C.byref(parts)), "flare_mlp_wgrad_partials")
    dev = g_out.device
    dwp = torch.empty(parts.value, L, Cdim, Cdim, dtype=torch.float32, device=dev)
    dbp = torch.empty(parts.value, L, Cdim, dtype=torch.float32, device=dev) if want_bias else None
    dw = torch.empty(L, Cdim, Cdim, dtype=torch.float32, device=dev)
    db = torch.empty(L, Cdim, dtype=torch.float32, device=dev) if want_bias else None
    with _on_device(dev):
        rows = 0 if gb is None and gb2 is None else (gb2 if gb is None else gb).shape[0]
        m, ws, off, splits = (None, None, 0, 0) if latents is None else latents
        rc = lib.flare_mlp_wgrad_block(C.byref(d), _ptr(a_in), T * Cdim if a_in.dim() == 3 else 0,
                                       _ptr(g_out), T * Cdim if g_out.dim() == 3 else 0, _ptr(dwp), _ptr(dbp), _ptr(dw), _ptr(db),
                                       _ptr(gb), _ptr(gb2), rows, _ptr(gsum), _ptr(gsum2), None if m is None else C.byref(m),
                                       None if ws is None else C.c_void_p(ws.data_ptr() + off), splits, 0 if dq is None else dq.shape[-1], _ptr(dq),
                                       C.c_void_p(_stream_ptr(dev)))
    _lib.check(rc, "flare_mlp_wgrad_block")
    return dw, db


class _FusedMlpFn(torch.autograd.Function):
    """y = res + chain(norm(x)); parameters are passed as inputs so that autograd routes their gradients:
    (x, res, gamma, beta, w_0 .. w_{L-1}, b_0 .. b_{L-1}) with None where a tensor does not exist."""

    @staticmethod
    def forward(ctx, mod, cd, norm, fmt, x, res, gamma, beta, *wb):
        out_dtype, x_head = fmt
        with torch.no_grad():
            ctx.operands = _train_operands(x, mod, cd)
            y = _fused_mlp_fwd(x, mod, cd, norm=norm, res=res, out_dtype=out_dtype, x_head=x_head, train=True, operands=ctx.operands)
        ctx.mod, ctx.cd, ctx.norm, ctx.x_head = mod, cd, norm, x_head
        # res and x one tensor: dy is added to dx inside the kernel.  (Two tensors over the same memory are not
        # enough: one of them may be detached, and then its path carries no gradient.)
        ctx.res_is_x = res is x
        ctx.has_res = res is not None
        ctx.n_wb = len(wb)
        # the backward reads the packed copies that the forward read, also where the module has other parameters by then (as after
        # torch.func.functional_call); as with a saved tensor, changing a parameter in place in between is an error
        ctx.versions = tuple(None if t is None else t._version for t in (gamma, beta, *wb))
        ctx.params = (gamma, beta, *wb)
        ctx.save_for_backward(x)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        (x,) = ctx.saved_tensors
        if ctx.versions != tuple(None if t is None else t._version for t in ctx.params):
            raise RuntimeError("a parameter of the fused MLP was modified in place between its forward and its backward")
        mod, cd, norm = ctx.mod, ctx.cd, ctx.norm
        if not ctx.x_head and _expand_factor(mod, x.shape[-1]):
            return _backward_expand(ctx, dy, x, _expand_factor(mod, x.shape[-1]))
        dx, gsum, dW, db, layers = _chain_backward(mod, cd, norm, x, dy, ctx.res_is_x, x_head=ctx.x_head, operands=ctx.operands, vectors=ctx.params[:2])
        L = len(layers)
        need = ctx.needs_input_grad            # (mod, cd, norm, fmt, x, res, gamma, beta, *wb)
        grads = [None, None, None, None]
        grads.append(dx.view(x.shape) if need[4] else None)
        grads.append(None if (not ctx.has_res or ctx.res_is_x or not need[5]) else dy)
        grads += _norm_grads(norm, gsum, need[6], need[7])
        for i, l in enumerate(layers):
            grads.append(dW[i].to(l.weight.dtype) if need[8 + i] else None)
        for i, l in enumerate(layers):
            grads.append(db[i].to(l.bias.dtype) if (l.bias is not None and need[8 + L + i]) else None)
        return tuple(grads)


def _norm_grads(norm, gsum, need_gamma, need_beta):
    if gsum is None:
        return [None, None]
    return [gsum[0].to(norm.weight.dtype) if need_gamma else None,
            gsum[1].to(norm.bias.dtype) if (need_beta and getattr(norm, "bias", None) is not None) else None]


def _chain_backward(mod, cd, norm, x, dy, res_is_x, dx_acc=None, x_head=0, operands=None, vectors=None):
    """Backward of y = [x +] chain(norm(x)) for the chain of C x C layers: (dx [T,C], the norm's [2,C] sums or None,
    dW [L,out,in], db [L,C] or None, the layers).  dx_acc: a [T,C] gradient of the same x that another chain left
    (x's dtype, contiguous); the kernel adds its result into it and it is returned as dx.  x_head: rows of x and dx hold padded
    heads (few tokens only).  operands, vectors: what the forward read, of the stack and of the norm."""
    lib = _lib.load()
    layers, act_mask, add_mask, act = _layers_of(mod)
    L = len(layers)
    Cdim, xw = layers[0].in_features, x.shape[-1]
    x = x.reshape(-1, xw)
    few = _few(x.shape[0], Cdim, L)
    operands = _train_operands(x, mod, cd) if operands is None else operands
    if len(operands) == 3:
        w_img, b, wt_img = operands          # the tiled operands
    elif x_head:
        raise RuntimeError("head-padded rows have a backward in the few-token launches only")
    else:
        few = 0
        _, b, w_img, wt_img = operands
    x2 = x
    x2 = _grid_rows(x2)
    dy2 = _rows2d(dy, Cdim)
    T = x2.shape[0]
    dev = x.device
    d = _lib.FlareMlpDesc()
    d.T, d.C, d.L = T, Cdim, L
    d.w_dtype, d.x_dtype, d.y_dtype = _dtype_code(w_img), _dtype_code(x2), _dtype_code(dy2)
    d.act, d.act_mask, d.add_mask = act, act_mask, add_mask
    d.x_stride, d.y_stride = x2.stride(0), dy2.stride(0)
    d.flags = (x_head // 4) << 8
    gamma, beta = _norm_args(d, norm, x, Cdim, vectors)
    if dx_acc is not None and (dx_acc.shape != (T, Cdim) or dx_acc.dtype != x2.dtype or not dx_acc.is_contiguous()):
        raise ValueError("dx_acc must be a contiguous [T, C] tensor of x's dtype")
    dx = dx_acc if dx_acc is not None else torch.empty(T, xw, dtype=x2.dtype, device=dev)
    a_in, g_out = (torch.empty(L, T, Cdim, dtype=cd, device=dev) for _ in range(2))
    dn = stats = gb = gsum = None
    any_bias = any(l.bias is not None for l in layers)
    if few and d.norm:
        gb = torch.empty(few, 2, Cdim, dtype=torch.float32, device=dev)
        gsum = torch.empty(2, Cdim, dtype=torch.float32, device=dev)
    elif d.norm:
        rows = C.c_int32(0)
        _lib.check(lib.flare_mlp_bwd_partial_rows(C.byref(d), C.byref(rows)), "flare_mlp_bwd_partial_rows")
        dn = torch.empty(T, Cdim, dtype=cd, device=dev)
        stats = torch.empty(T, 2, dtype=torch.float32, device=dev)
        gb = torch.empty(rows.value, 2, Cdim, dtype=torch.float32, device=dev)
        gsum = torch.empty(2, Cdim, dtype=torch.float32, device=dev)
    bits = (_lib.MLP_BWD_ADD_DY if res_is_x else 0) | (_lib.MLP_BWD_ACCUMULATE if dx_acc is not None else 0)
    with _on_device(dev):
        if few:
            rc = lib.flare_mlp_few_bwd(C.byref(d), _ptr(x2), _ptr(dy2), None, _ptr(w_img), _ptr(wt_img), _ptr(b), _ptr(gamma), _ptr(beta),
                                       bits, _ptr(dx), _ptr(a_in), _ptr(g_out), _ptr(gb), C.c_void_p(_stream_ptr(dev)))
        else:
            rc = lib.flare_mlp_bwd(C.byref(d), _ptr(x2), _ptr(dy2), _ptr(w_img), _ptr(wt_img), _ptr(b), _ptr(gamma), _ptr(beta),
                                   bits, _ptr(dx), _ptr(a_in), _ptr(g_out), _ptr(dn), _ptr(stats), _ptr(gb),
                                   None, C.c_void_p(_stream_ptr(dev)))
    _lib.check(rc, "flare_mlp_bwd")
    # weight and bias gradients: one more launch over the rows the kernel left (16-bit products with fp32
    # accumulation, as torch runs a Linear's backward under autocast); norm gradients: partial rows, summed with the others
    dW, db = _weight_grads(d, g_out, a_in, any_bias, gb=gb, gsum=gsum)                 # [L, out, in], [L, C] fp32
    return dx, gsum, dW, db, layers


def _pair_backward(mod_a, mod_b, cd, norm, x, dya, dyb, operands, vectors, y_head=0, dres=None, into=None):
    """Backward of both stacks of a pair in one launch (operands, vectors: what the forward read, of the stacks and of the norm; y_head: dya
    and dyb are rows of padded heads; dres: another gradient of x, added to dx): (dx, the norm's [2,C] sums or None, dW [2L,out,in], db [2L,C] or
    None, the 2 L layers)."""
    lib = _lib.load()
    layers, act_mask, add_mask, act = _pair_info(x, mod_a, mod_b, cd)
    w, b, wt = operands
    L2, Cdim, dev = len(layers), x.shape[-1], x.device
    x2 = x.reshape(-1, Cdim)
    x2 = _grid_rows(x2)
    yw = Cdim // y_head * 16 if y_head else Cdim
    da, db_ = _rows2d(dya, yw), _rows2d(dyb, yw)
    if da.dtype != db_.dtype:
        da, db_ = da.float(), db_.float()
    if da.stride() != db_.stride():
        da, db_ = da.contiguous(), db_.contiguous()
    T = x2.shape[0]
    d = _lib.FlareMlpDesc()
    d.T, d.C, d.L = T, Cdim, L2 // 2
    d.w_dtype, d.x_dtype, d.y_dtype = _dtype_code(w), _dtype_code(x2), _dtype_code(da)
    d.act, d.act_mask, d.add_mask = act, act_mask, add_mask
    d.x_stride, d.y_stride = x2.stride(0), da.stride(0)
    d.flags = (y_head // 4) << 12
    gamma, beta = _norm_args(d, norm, x, Cdim, vectors)
    dx = torch.empty(T, Cdim, dtype=x2.dtype, device=dev)
    rows = torch.empty(2, L2, T, Cdim, dtype=cd, device=dev) if into is None else into         # a_in, g_out
    gb = gsum = None
    if d.norm:
        gb = torch.empty(_few(T, Cdim, L2 // 2), 2, Cdim, dtype=torch.float32, device=dev)
        gsum = torch.empty(2, Cdim, dtype=torch.float32, device=dev)
    r2 = None
    if dres is not None:
        r2 = dres.reshape(-1, Cdim)
        if r2.dtype != x2.dtype or not r2.is_contiguous() or r2.data_ptr() % 16:
            r2 = r2.to(x2.dtype, copy=True, memory_format=torch.contiguous_format)
    with _on_device(dev):
        rc = lib.flare_mlp_few_bwd_res(C.byref(d), _ptr(x2), _ptr(da), _ptr(db_), _ptr(r2), _ptr(w), _ptr(wt), _ptr(b), _ptr(gamma),
                                       _ptr(beta), 0, _ptr(dx), _ptr(rows[0]), _ptr(rows[1]), _ptr(gb), C.c_void_p(_stream_ptr(dev)))
    _lib.check(rc, "flare_mlp_few_bwd_res")
    if into is not None:                       # (dx, the norm's partial rows or None): the caller forms the weight gradients
        return dx, gb
    dW, db = _weight_grads(d, rows[1], rows[0], any(l.bias is not None for l in layers), gb=gb, gsum=gsum)
    return dx, gsum, dW, db, layers


class _FusedPairFn(torch.autograd.Function):
    """(ya, yb) = (chain_a(norm(x)), chain_b(norm(x))): two chains that read the same rows through the same norm (the k
    and v projections of a block).  Forward: the two launches of _FusedMlpFn.  Backward: the second chain's launch adds
    its gradient of x into the first one's, which autograd would otherwise do with a launch of its own over three
    [T, C] arrays.  Inputs: (x, gamma, beta, weights and biases of a, weights and biases of b)."""

    @staticmethod
    def forward(ctx, mod_a, mod_b, cd, norm, fmt, x, gamma, beta, *wb):
        out_dtype, y_head, with_res = fmt
        with torch.no_grad():
            info = _pair_info(x, mod_a, mod_b, cd)
            packed = None if info is None else _packed_few(mod_a, info[0], cd, True)
            ctx.pair = packed is not None
            n = len(info[0]) // 2 if ctx.pair else 0
            if y_head and not ctx.pair:
                raise ValueError("head-padded rows have no backward here: call under torch.no_grad()")
            pair = [] if ctx.pair else None
            a, b = (((packed[0][:n], packed[1][:n]), (packed[0][n:], packed[1][n:])) if ctx.pair else
                    (_train_operands(x, mod_a, cd), _train_operands(x, mod_b, cd)))
            ya = _fused_mlp_fwd(x, mod_a, cd, norm=norm, out_dtype=out_dtype, y_head=y_head, train=True, operands=a, pair=pair)
            yb = _fused_mlp_fwd(x, mod_b, cd, norm=norm, out_dtype=out_dtype, y_head=y_head, train=True, operands=b, pair=pair)
        ctx.operands = packed if ctx.pair else (a, b)
        ctx.mods, ctx.cd, ctx.norm, ctx.y_head = (mod_a, mod_b), cd, norm, y_head
        ctx.versions = tuple(None if t is None else t._version for t in (gamma, beta, *wb))
        ctx.params = (gamma, beta, *wb)
        ctx.save_for_backward(x)
        return (ya, yb, x.view_as(x)) if with_res else (ya, yb)

    @staticmethod
    @once_differentiable
    def backward(ctx, dya, dyb, dres=None):
        (x,) = ctx.saved_tensors
        if ctx.versions != tuple(None if t is None else t._version for t in ctx.params):
            raise RuntimeError("a parameter of the fused MLP was modified in place between its forward and its backward")
        mod_a, mod_b = ctx.mods
        if ctx.pair:
            dx, gs, dW, db, layers = _pair_backward(mod_a, mod_b, ctx.cd, ctx.norm, x, dya, dyb, ctx.operands, ctx.params[:2], ctx.y_head, dres)
            n = len(layers) // 2
            la, lb, dWa, dWb = layers[:n], layers[n:], dW[:n], dW[n:]
            dba, dbb = (None, None) if db is None else (db[:n], db[n:])
        else:
            (a, b), vectors = ctx.operands, ctx.params[:2]
            dx, gs_a, dWa, dba, la = _chain_backward(mod_a, ctx.cd, ctx.norm, x, dya, False, operands=a, vectors=vectors)
            dx, gs_b, dWb, dbb, lb = _chain_backward(mod_b, ctx.cd, ctx.norm, x, dyb, False, dx_acc=dx, operands=b, vectors=vectors)
            gs = None if gs_a is None else gs_a + gs_b
        need = ctx.needs_input_grad            # (mod_a, mod_b, cd, norm, fmt, x, gamma, beta, *wb)
        grads = [None, None, None, None, None, dx.view(x.shape) if need[5] else None]
        grads += _norm_grads(ctx.norm, gs, need[6], need[7])
        at = 8
        for layers, dW, db in ((la, dWa, dba), (lb, dWb, dbb)):
            n = len(layers)
            for i, l in enumerate(layers):
                grads.append(dW[i].to(l.weight.dtype) if need[at + i] else None)
            for i, l in enumerate(layers):
                grads.append(db[i].to(l.bias.dtype) if (l.bias is not None and need[at + n + i]) else None)
            at += 2 * n
        return tuple(grads)


def _rows2d(t, Cdim):
    t2 = t.reshape(-1, Cdim)
    if t2.dtype not in (torch.float32, torch.bfloat16, torch.float16):
        t2 = t2.float()
    return _grid_rows(t2)


def _backward_expand(ctx, dy, x, E):
    """Backward of y = res + fc2(act(fc1(norm(x)))) with hidden width E C: flare_mlp_expand_bwd, then two passes of
    flare_mlp_wgrad (dW1, db1 from the rows dt against n; dW2, db2 from dy against the rows h)."""
    mod, cd, norm = ctx.mod, ctx.cd, ctx.norm
    lib = _lib.load()
    _, _, _, act = _layers_of(mod)
    f1, f2 = mod.fc1, mod.fc2
    Cdim = x.shape[-1]
    _, b, w_img, wt_img = ctx.operands
    x2, dy2 = _rows2d(x, Cdim), _rows2d(dy, Cdim)
    T = x2.shape[0]
    dev = x.device
    d = _lib.FlareMlpDesc()
    d.T, d.C, d.L, d.flags = T, Cdim, 2 * E, _lib.MLP_EXPAND
    d.w_dtype, d.x_dtype, d.y_dtype = _dtype_code(w_img), _dtype_code(x2), _dtype_code(dy2)
    d.act, d.act_mask, d.add_mask = act, 1, 0
    d.x_stride, d.y_stride = x2.stride(0), dy2.stride(0)
    gamma, beta = _norm_args(d, norm, x, Cdim, ctx.params[:2])
    dx = torch.empty(T, Cdim, dtype=x2.dtype, device=dev)
    n_row = torch.empty(T, Cdim, dtype=cd, device=dev)
    dy_row = torch.empty(T, Cdim, dtype=cd, device=dev)
    h = torch.empty(E, T, Cdim, dtype=cd, device=dev)
    dt = torch.empty(E, T, Cdim, dtype=cd, device=dev)
    dn = stats = gb = gsum = None
    if d.norm:
        rows = C.c_int32(0)
        _lib.check(lib.flare_mlp_bwd_partial_rows(C.byref(d), C.byref(rows)), "flare_mlp_bwd_partial_rows")
        dn = torch.empty(T, Cdim, dtype=cd, device=dev)
        stats = torch.empty(T, 2, dtype=torch.float32, device=dev)
        gb = torch.empty(rows.value, 2, Cdim, dtype=torch.float32, device=dev)
        gsum = torch.empty(2, Cdim, dtype=torch.float32, device=dev)
    with _on_device(dev):
        rc = lib.flare_mlp_expand_bwd(C.byref(d), _ptr(x2), _ptr(dy2), _ptr(w_img), _ptr(wt_img), _ptr(b), _ptr(gamma), _ptr(beta),
                                      1 if ctx.res_is_x else 0, _ptr(dx), _ptr(n_row), _ptr(dy_row), _ptr(h), _ptr(dt),
                                      _ptr(dn), _ptr(stats), _ptr(gb), _ptr(gsum), C.c_void_p(_stream_ptr(dev)))
    _lib.check(rc, "flare_mlp_expand_bwd")
    dW1, db1 = _weight_grads(d, dt, n_row, f1.bias is not None)          # [E, C(hidden chunk), C(in)], [E, C]
    dW2, db2 = _weight_grads(d, dy_row, h, f2.bias is not None, L=E)     # [E, C(out), C(hidden chunk)], [E, C] (E equal rows)
    need = ctx.needs_input_grad            # (mod, cd, norm, fmt, x, res, gamma, beta, w1, w2, b1, b2)
    grads = [None, None, None, None]
    grads.append(dx.view(x.shape) if need[4] else None)
    grads.append(None if (not ctx.has_res or ctx.res_is_x or not need[5]) else dy)
    if d.norm:
        grads.append(gsum[0].to(norm.weight.dtype) if need[6] else None)
        grads.append(gsum[1].to(norm.bias.dtype) if (need[7] and getattr(norm, "bias", None) is not None) else None)
    else:
        grads += [None, None]
    grads.append(dW1.reshape(E * Cdim, Cdim).to(f1.weight.dtype) if need[8] else None)
    grads.append(dW2.permute(1, 0, 2).reshape(Cdim, E * Cdim).to(f2.weight.dtype) if need[9] else None)
    grads.append(db1.reshape(E * Cdim).to(f1.bias.dtype) if (f1.bias is not None and need[10]) else None)
    grads.append(db2[0].to(f2.bias.dtype) if (f2.bias is not None and need[11]) else None)
    return tuple(grads)


def _fused_mlp_train(x, mod, cd, norm, res, out_dtype, x_head=0):
    layers = _layers_of(mod)[0]
    has_norm = norm is not None and not isinstance(norm, nn.Identity)
    gamma = getattr(norm, "weight", None) if has_norm else None
    beta = getattr(norm, "bias", None) if has_norm else None
    wb = [l.weight for l in layers] + [l.bias for l in layers]
    return _FusedMlpFn.apply(mod, cd, norm if has_norm else None, (out_dtype, x_head), x, res, gamma, beta, *wb)
