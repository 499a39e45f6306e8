"""A FLAREBlock's inference forward as one call into the library.

Under autocast and without gradients the block is seven launches (norm + k projection, norm + v projection, three of the mixer,
output projection + residual, norm + feed-forward + residual; pdebench/models/flare.py:107-215), five on few tokens, where the two
projections and the block's end are one launch each.  On small point clouds enqueueing them from Python is what it costs: calls of
20 to 30 us each, most of it spent deciding again what the last call decided.  An 8-block model of 64 channels on 3973 points:
1070 us a forward, 340 us through the plans (0.24 ms of kernels).  `forward` keeps what depends on the module and the shape only --
descriptors, the packed 16-bit weights the modules hold anyway, the layout of one scratch allocation -- and hands the rest to
flare_block_fwd.  Nothing about an input is kept.

A block's first forward runs the general path of modules.py, which packs the weights; from then on a plan is made where a shape is
new.  Making one takes about as long as the general path's own decisions, so that a loop over meshes of ever new sizes is no
slower for it (us a forward of the 8 blocks, 1000 to 5000 points, general path / plans: a new size every time 1082 / 986, the next
forward of that size 1082 / 400, nine sizes in turn 1036 / 325, weights changed before every forward 2290 / 2100).

Every call compares what the block's plans were made from: the modules' structure, every parameter's address and version, the norms' eps,
the mixer's scale.  Where any of it changed, all plans of the block go, whatever their shape.  The parameters' memory is held as long as
plans name its address: another tensor put in a parameter's place then always lies elsewhere.  Calls a plan does not cover (hooks on the
attention module, gradients, rows off the 16-byte grid, head dims or latent counts that the mixer pads itself) run the general path.
No plan is made while a graph is recorded: the packing of k and v would be recorded too, and a call before the first replay would read
weights that nothing has written yet.
"""
from __future__ import annotations

import ctypes as C

import torch
from torch import nn

from . import _lib, functional, fused, rows

_MAX_SHAPES = 32          # plans kept per block, the newest; a plan holds a descriptor of 0.5 KB and references to packed weights, which all
                          # plans of a block share (one packing for few tokens, one for many)
_X_DTYPES = (torch.float32, torch.bfloat16, torch.float16)


class _Plans(dict):
    """shape -> plan, or False where the general path serves it; all made from the module as `key` describes it (None before the first).
    held: the parameters' memory, whose addresses are in the key.  pair: compute type -> joint packing of the k and v projections.
    Never changed to another key: a block whose key differs gets another object, so that a plan under way in one thread cannot join
    the plans that another thread began.
    A copy of a module, and one read back from a file, begins without plans: they hold addresses."""

    def __init__(self, key=None, held=()):
        super().__init__()
        self.key, self.held, self.pair = key, held, {}

    def __deepcopy__(self, memo):
        return _Plans()

    def __reduce__(self):
        return _Plans, ()


class _Plan:
    __slots__ = ("desc", "ref", "scratch", "keep")


def _parameters(block):
    """The parameters whose addresses are in the block's key (without a walk over the modules, which is slower than the rest of a plan)."""
    m, a = block._modules, block._modules["att"]._modules
    owners = [m["att"], m["norm1"], m["norm2"]]
    for mod in (a["k_proj"], a["v_proj"], a["out_proj"], m["mlp"]):
        owners += fused._layers_of(mod)[0]
    return [t for o in owners for t in o._parameters.values() if t is not None]


def _key(block):
    """Everything a plan is made from, or None for a block that the general path serves."""
    m = block._modules
    att, mlp, n1, n2 = (m.get(name) for name in ("att", "mlp", "norm1", "norm2"))
    if mlp is None or n1 is None or n2 is None or not rows._plain(att) or att.qk_norm or "latent_q" not in att._parameters:
        return None
    a = att._modules
    layers, key = [], [att.attn_scale, att.num_heads, att.num_latents, att.head_dim]
    for mod in (a["k_proj"], a["v_proj"], a["out_proj"], mlp):
        info = fused._layers_of(mod)
        if info is None:
            return None
        key.append(fused._structure_key(mod))
        layers += info[0]
    for n in (n1, n2):
        p = n._parameters
        for name in ("weight", "bias"):
            t = p.get(name)
            key.append(None if t is None else (t.data_ptr(), t._version))
        key += (type(n), getattr(n, "eps", None))
    if any("weight" not in l._parameters or "bias" not in l._parameters for l in layers):      # parametrised: another tensor at every access
        return None
    q = att._parameters["latent_q"]
    key.append((q.data_ptr(), q._version))
    key.append(fused._param_key(layers))
    return key


def _mlp(mod, T, cd, x_dtype, y_dtype, x_stride, y_stride, norm=None, res=None, x_head=0, y_head=0, operands=None):
    """(descriptor, weights, biases, gamma, beta) of one launch of fused._fused_mlp_fwd, or None.  operands: this stack's part of a
    joint few-token packing."""
    info, io, Cdim, E = fused._forward_plan(mod)
    layers, act_mask, add_mask, act = info
    if io is not None or (E and (x_head or y_head)):
        return None
    few = operands is not None
    w, b = operands if few else (None, None)
    if not few and not E and fused._few(T, Cdim, len(layers)):
        packed = fused._packed_few(mod, layers, cd, False)
        if packed is not None:
            few, (w, b) = True, packed[:2]
    if w is None:
        w, b = fused._packed_expand(mod, E, cd) if E else fused._packed(mod, layers, cd)
    if E:
        act_mask, add_mask = 1, 0
    d = _lib.FlareMlpDesc()
    d.T, d.C, d.L = T, Cdim, w.shape[0]
    d.flags = (_lib.MLP_EXPAND if E else _lib.MLP_W_TILED if few else 0) | ((x_head // 4) << 8) | ((y_head // 4) << 12)
    d.w_dtype, d.x_dtype, d.y_dtype = functional._DTYPES[cd], functional._DTYPES[x_dtype], functional._DTYPES[y_dtype]
    d.act, d.act_mask, d.add_mask, d.x_stride, d.y_stride = act, act_mask, add_mask, x_stride, y_stride
    gamma = beta = None
    if norm is not None:
        gamma, beta = norm._parameters.get("weight"), norm._parameters.get("bias")
        if gamma is None or any(t is not None and fused._vec32(t) is not t for t in (gamma, beta)):
            return None                                   # a converted copy would have to follow its parameter
        fused._norm_args(d, norm, torch.empty(0, dtype=x_dtype), Cdim)
    if res is not None:
        d.res_dtype, d.res_stride = functional._DTYPES[res], Cdim
    return d, w, b, gamma, beta


def _build(block, x, cd, plans):
    """A plan for inputs of x's shape and type, or None where the general path has to serve them."""
    att, mlp = block.att, block.mlp
    B, N, Cdim = x.shape
    H, M, D = att.num_heads, att.num_latents, att.head_dim
    if any(fused.compute_dtype(x, m) is not cd for m in (att.k_proj, att.v_proj, att.out_proj, mlp)):
        return None
    if M % 32 or D not in (4, 8, 16, 32, 64) or any(type(n) not in (nn.LayerNorm, nn.RMSNorm) for n in (block.norm1, block.norm2)):
        return None
    dev = x.device
    if any(p.device != dev for p in _parameters(block)):
        return None
    head = D if D in (4, 8) else 0                        # narrow heads: k, v and the mixer's rows padded to 16 columns
    Dp, T = (16 if head else D), B * N
    width = H * Dp
    # few tokens: the projections' weights in one piece, so that one launch serves both
    info, kv = fused._pair_info(x, att.k_proj, att.v_proj, cd), (None, None)
    if info is not None:
        if cd not in plans.pair:
            tiles = fused._chain_tiles(info[0])
            plans.pair[cd] = None if tiles is None else fused._pack_launch(Cdim, cd, tiles, x.device, False, tiled=True)
        packed = plans.pair[cd]
        if packed is not None:
            n = len(info[0]) // 2
            kv = (packed[0][:n], packed[1][:n]), (packed[0][n:], packed[1][n:])
    parts = [_mlp(att.k_proj, T, cd, x.dtype, cd, Cdim, width, norm=block.norm1, y_head=head, operands=kv[0]),
             _mlp(att.v_proj, T, cd, x.dtype, cd, Cdim, width, norm=block.norm1, y_head=head, operands=kv[1]),
             _mlp(att.out_proj, T, cd, cd, x.dtype, width, Cdim, res=x.dtype, x_head=head),
             _mlp(mlp, T, cd, x.dtype, x.dtype, Cdim, Cdim, norm=block.norm2, res=x.dtype)]
    if any(p is None for p in parts):
        return None
    q = att._cached_q(cd, Dp - D)
    plan = _Plan()
    d = plan.desc = _lib.FlareBlockDesc()
    for i, (desc, w, b, gamma, beta) in enumerate(parts):
        d.mlp[i], d.w[i], d.b[i] = desc, w.data_ptr(), b.data_ptr()
        d.gamma[i], d.beta[i] = (None if t is None else t.data_ptr() for t in (gamma, beta))
    d.q = q.data_ptr()
    m = d.mixer
    m.B, m.H, m.N, m.M, m.D, m.dtype, m.scale, m.flags = B, H, N, M, Dp, functional._DTYPES[cd], float(att.attn_scale), functional._extra_mixer_flags
    m.q_stride = _lib.I3(0, M * Dp, Dp)
    m.k_stride = m.v_stride = m.y_stride = _lib.I3(N * width, Dp, width)
    n = C.c_size_t(0)
    if _lib.load().flare_block_scratch_bytes(C.byref(d), C.byref(n)) != _lib.FLARE_OK:
        return None
    plan.ref, plan.scratch = C.byref(d), n.value
    plan.keep = [q] + [t for p in parts for t in p[1:]]   # the parameters' packed copies, and the norms' vectors
    return plan


def forward(block, x):
    """block(x) through a plan, or None: the general path serves the call."""
    if torch.is_grad_enabled() or type(x) is not torch.Tensor or not x.is_cuda or not torch.is_autocast_enabled("cuda"):
        return None
    cd = torch.get_autocast_dtype("cuda")
    if (cd not in (torch.bfloat16, torch.float16) or x.dtype not in _X_DTYPES or x.dim() != 3 or x.numel() == 0
            or not x.is_contiguous() or x.data_ptr() % 16):
        return None
    plans = block.__dict__.get("_flare_plans")
    if plans is None:
        block.__dict__["_flare_plans"] = _Plans()
        return None
    key = _key(block)
    if key is None:
        return None
    dev = x.device
    shape = (x.shape, x.dtype, cd, dev.index, functional._extra_mixer_flags)
    plan = plans.get(shape) if plans.key == key else None
    if plan is None:
        if torch.cuda.is_current_stream_capturing():
            return None
        if plans.key != key:
            plans = block.__dict__["_flare_plans"] = _Plans(key, [fused.hold(t) for t in _parameters(block)])
        for oldest in list(plans)[:len(plans) + 1 - _MAX_SHAPES]:
            plans.pop(oldest, None)
        plan = plans[shape] = _build(block, x, cd, plans) or False
    if not plan:
        return None
    y = torch.empty_like(x)
    scratch = torch.empty(plan.scratch, dtype=torch.uint8, device=dev)
    with functional._on_device(dev):
        rc = _lib.load().flare_block_fwd(plan.ref, x.data_ptr(), y.data_ptr(), scratch.data_ptr(), plan.scratch, functional._stream_ptr(dev))
    if rc:
        _lib.check(rc, "flare_block_fwd")
    return y
