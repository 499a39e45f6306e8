"""A FLAREBlock's training step on few tokens as one autograd node.

On small meshes a step is the sum of its launches' latencies.  The block's four token-wise launches and the mixer
(pdebench/models/flare.py:107-215) run as in modules.py; what one node for all of them saves is launches: the rows that the
backward leaves for the weight gradients lie side by side, so that one product launch and one launch of sums serve every
layer, both norms and the latents of the block, instead of one each per stack; the output projection and the feed-forward are one
launch each way; the latents are cast by the packing launch.  Replayed training step of 8 blocks, 4096 points, bf16: 128 channels
1518 -> 1342 (weight gradients) -> 1261 (the block's end) -> 1238 (two workgroups of the forward on a CU) -> 1208 us (latents), 64
channels 1171 -> 1024 -> 966 -> 966 -> 894 us (1178 and 873 us since the mixer's small launches spread over the chip).

Used under autocast with gradients enabled, where all stacks are plain chains that the few-token launches take, the parameters can be read
by the packing launch, and nothing hooks into the attention module; `forward` answers None for every other call.
"""
from __future__ import annotations

import ctypes as C

import torch
from torch import nn
from torch.autograd.function import once_differentiable

from . import _lib, functional, fused, rows


def _stacks(block):
    att = block.att
    return att.k_proj, att.v_proj, att.out_proj, block.mlp


def _plan(block, x, cd):
    """(layers of k, v, out and mlp in that order; columns of a head in the mixer) or None."""
    att = block.att
    k, v, out, mlp = _stacks(block)
    B, N, Cdim = x.shape
    H, M, D = att.num_heads, att.num_latents, att.head_dim
    if M % 32 or D not in (4, 8, 16, 32, 64) or any(fused.compute_dtype(x, m) is not cd for m in (k, v, out, mlp)):
        return None
    info, chain = fused._pair_info(x, k, v, cd), fused._layers_of(mlp)
    if info is None or not isinstance(out, nn.Linear) or fused._expand_factor(mlp, Cdim) or any(fused._train_subchain(m) is not None for m in (k, v, mlp)):
        return None
    layers = info[0] + [out] + chain[0]
    if len(chain[0]) > fused._BWD_MAX_LAYERS[Cdim] or len(layers) > _lib.MLP_PACK_MAX:
        return None
    Dp = 16 if D < 16 else D
    d = _lib.FlareMixerDesc()
    d.B, d.H, d.N, d.M, d.D, d.dtype, d.scale, d.flags = B, H, N, M, Dp, functional._DTYPES[cd], 1.0, functional._extra_mixer_flags
    d.q_stride = _lib.I3(0, M * Dp, Dp)
    d.k_stride = d.v_stride = d.y_stride = _lib.I3(N * H * Dp, Dp, H * Dp)
    n = C.c_size_t(0)
    if _lib.load().flare_mixer_bwd_workspace_bytes(C.byref(d), C.byref(n)) != _lib.FLARE_OK or fused._chain_tiles(layers) is None:
        return None
    return layers, Dp


class _BlockFn(torch.autograd.Function):
    """Inputs: (block, compute type, layers, columns of a head, x, latent_q, norm weights and biases, the layers' weights, their biases)."""

    @staticmethod
    def forward(ctx, block, cd, layers, Dp, x, latent_q, g1, b1, g2, b2, *wb):
        att = block.att
        k, v, out, mlp = _stacks(block)
        B, N, _ = x.shape
        H, M, D = att.num_heads, att.num_latents, att.head_dim
        head = D if Dp != D else 0
        with torch.no_grad():
            q = latent_q.view(H, M, D)
            q16 = torch.empty(H, M, Dp, dtype=cd, device=x.device) if fused._readable(q) and q.is_contiguous() and q.device == x.device else None
            if not fused.prepack(x, cd, (k, v), (out,), (mlp,), latents=None if q16 is None else (q, q16)) or q16 is None:
                q16 = torch.nn.functional.pad(q.to(cd), (0, Dp - D)) if head else q.to(cd)
            n = (len(layers) - 1 - len(fused._layers_of(mlp)[0])) // 2
            ctx.operands = fused._packed_few(k, layers[:2 * n], cd, True), fused.tail_operands(out, mlp, cd)
            w, b = ctx.operands[0][:2]
            pair = []
            k2 = fused._fused_mlp_fwd(x, k, cd, norm=block.norm1, out_dtype=cd, y_head=head, train=True, operands=(w[:n], b[:n]), pair=pair)
            v2 = fused._fused_mlp_fwd(x, v, cd, norm=block.norm1, out_dtype=cd, y_head=head, train=True, operands=(w[n:], b[n:]), pair=pair)
            kh, vh = (t.view(B, N, H, Dp).permute(0, 2, 1, 3) for t in (k2, v2))
            y, z, lse_lat, lse_tok = functional._mixer_forward(q16, kh, vh, float(att.attn_scale), None, 0, False, True, True)
            y2 = y.permute(0, 2, 1, 3).reshape(B, N, H * Dp)
            x1, o = fused.tail_forward(y2, out, x, mlp, cd, block.norm2, head, ctx.operands[1])
        ctx.block, ctx.cd, ctx.layers, ctx.n, ctx.head, ctx.scale = block, cd, layers, n, head, float(att.attn_scale)
        ctx.dims, ctx.norms = (B, N, H, Dp, D), (block.norm1, block.norm2)
        # the backward reads the packed copies that the forward read, also where the block has other parameters by then; as with a saved
        # tensor, changing one in place before is an error (of the latents it reads the saved copy, which stays as it was)
        ctx.q_like, ctx.params = latent_q, (g1, b1, g2, b2, *wb)
        ctx.versions = tuple(None if t is None else t._version for t in ctx.params)
        ctx.save_for_backward(x, k2, v2, q16, y2, z, lse_lat, lse_tok, x1)
        return o

    @staticmethod
    @once_differentiable
    def backward(ctx, do):
        x, k2, v2, q16, y2, z, lse_lat, lse_tok, x1 = (t.contiguous() for t in ctx.saved_tensors)      # hooks may have changed their order
        if ctx.versions != tuple(None if t is None else t._version for t in ctx.params):
            raise RuntimeError("a parameter of the block was modified in place between its forward and its backward")
        block, cd, layers, n, head = ctx.block, ctx.cd, ctx.layers, ctx.n, ctx.head
        k, v, out, mlp = _stacks(block)
        B, N, H, Dp, D = ctx.dims
        Cdim, T, L, dev = x.shape[-1], B * N, len(layers), x.device
        norm1, norm2 = ctx.norms
        a_in, g_out = torch.empty(2, L, T, Cdim, dtype=cd, device=dev)
        m = 2 * n
        vectors = ctx.params
        dx1, dy, gb2 = fused.tail_backward(y2, out, x1, mlp, cd, norm2, head, do, a_in[m:], g_out[m:], ctx.operands[1], vectors[2:4])
        kh, vh, yh, gyh = (t.view(B, N, H, Dp).permute(0, 2, 1, 3) for t in (k2, v2, y2, dy))
        latents, dk, dv = functional._mixer_hip_grad(q16, kh, vh, yh, z, lse_lat, lse_tok, ctx.scale, gyh, dq_parts=True)
        dq = torch.empty(H, q16.shape[1], D, dtype=torch.float32, device=dev)
        dk, dv = (t.permute(0, 2, 1, 3).reshape(T, H * Dp) for t in (dk, dv))
        dx, gb1 = fused._pair_backward(k, v, cd, norm1, x, dk, dv, ctx.operands[0], vectors[:2], head, dx1, into=(a_in[:m], g_out[:m]))
        gs1, gs2 = (None if g is None else torch.empty(2, Cdim, dtype=torch.float32, device=dev) for g in (gb1, gb2))
        d = _lib.FlareMlpDesc()
        d.w_dtype = functional._DTYPES[cd]
        dW, db = fused._weight_grads(d, g_out, a_in, any(l.bias is not None for l in layers), gb=gb1, gsum=gs1, gb2=gb2, gsum2=gs2, latents=latents, dq=dq)
        need = ctx.needs_input_grad            # (block, cd, layers, Dp, x, latent_q, g1, b1, g2, b2, *wb)
        q_like = ctx.q_like
        grads = [None, None, None, None, dx.view(x.shape) if need[4] else None,
                 dq.reshape(q_like.shape).to(q_like.dtype) if need[5] else None]
        for norm, gs, at in ((norm1, gs1, 6), (norm2, gs2, 8)):
            grads += fused._norm_grads(norm, gs, need[at], need[at + 1])
        grads += [dW[i].to(l.weight.dtype) if need[10 + i] else None for i, l in enumerate(layers)]
        grads += [db[i].to(l.bias.dtype) if l.bias is not None and need[10 + L + i] else None for i, l in enumerate(layers)]
        return tuple(grads)


def forward(block, x):
    """block(x) as one node, or None: the general path serves the call."""
    Cdim = x.shape[-1]
    if (not torch.is_grad_enabled() or type(x) is not torch.Tensor or not x.is_cuda or x.dim() != 3
            or not 0 < x.numel() // Cdim <= fused._FEW_TOKENS.get(Cdim, 0) or not torch.is_autocast_enabled("cuda")):
        return None
    cd, att = torch.get_autocast_dtype("cuda"), block.att
    if (cd not in (torch.bfloat16, torch.float16) or not x.is_contiguous() or x.data_ptr() % 16 or att.qk_norm or not rows._plain(att)
            or x.dtype not in (torch.float32, torch.bfloat16, torch.float16) or type(att.latent_q) is not nn.Parameter):
        return None
    plan = _plan(block, x, cd)
    if plan is None:
        return None
    norms = [n if isinstance(n, (nn.LayerNorm, nn.RMSNorm)) else None for n in (block.norm1, block.norm2)]
    if any(n is None for n in norms):
        return None
    layers, Dp = plan
    nb = [t for n in norms for t in (n.weight, getattr(n, "bias", None))]
    return _BlockFn.apply(block, cd, layers, Dp, x, att.latent_q, *nb, *(l.weight for l in layers), *(l.bias for l in layers))
