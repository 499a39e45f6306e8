"""Functional API of the MI355X FLARE engine.

Mirrors the reference's operator interface (paths relative to the reference tree):
  flare_multihead_mixer(q, k, v)          README.md:39-52
  TripleAttentionFunction.apply(...)      lra/models/triton/triple.py:27-121 -> (STATE, O)
and adds the entry points the causal path needs (flare_causal_prefill / _decode).

Every function here launches HIP kernels from libflare_hip.so through ctypes.  torch is
used for device memory, streams and autograd plumbing only; there is no PyTorch or CPU
implementation behind these calls, and a missing library raises.
"""
from __future__ import annotations

import ctypes as C
import struct
import math
from typing import Optional, Tuple

import torch
from torch.autograd.function import once_differentiable

from . import _lib
from ._lib import FlareCausalDesc, FlareMixerDesc, FlareTripleDesc

_DTYPES = {torch.float32: _lib.DT_F32, torch.bfloat16: _lib.DT_BF16, torch.float16: _lib.DT_F16}


def _dtype_code(t: torch.Tensor) -> int:
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}; expected float32, bfloat16 or float16") from None


def _require_cuda(*ts: torch.Tensor):
    dev = ts[0].device
    for t in ts:
        if t.device.type != "cuda":
            raise RuntimeError(
                "FLARE HIP kernels need tensors on a HIP device ('cuda'); got "
                f"{t.device}. There is no CPU implementation in this package.")
        if t.device != dev:
            raise RuntimeError("all tensors must live on the same device")


def _rows_last_contig(t: torch.Tensor) -> torch.Tensor:
    """[B,H,N,D] tensor usable without a copy iff its innermost stride is 1."""
    if t.stride(-1) != 1 and t.size(-1) != 1:
        return t.contiguous()
    return t


def _s3(t: torch.Tensor):
    """(b, h, row) element strides of a 4-d tensor."""
    return _lib.I3(t.stride(0), t.stride(1), t.stride(2))


def _q4(q: torch.Tensor, B: int) -> torch.Tensor:
    """Latent queries as a [B?,H,M,D] view; a 3-d q is shared over the batch (stride 0)."""
    if q.dim() == 3:
        q = q.unsqueeze(0).expand(B, -1, -1, -1)
    elif q.dim() != 4:
        raise ValueError(f"q must be [H,M,D] or [B,H,M,D], got shape {tuple(q.shape)}")
    if q.stride(-1) != 1 and q.size(-1) != 1:
        q = q.contiguous()
    return q


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream_ptr(dev) -> int:
    """The HIP stream torch would launch on for this device (every launch of the library goes there)."""
    if _raw_stream is not None:          # the same handle without building a torch.cuda.Stream object per call
        idx = dev.index if isinstance(dev, torch.device) else dev
        return _raw_stream(torch.cuda.current_device() if idx is None else idx)
    return torch.cuda.current_stream(dev).cuda_stream


class _NoGuard:
    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


_NO_GUARD = _NoGuard()


def _on_device(dev):
    """Context that makes dev the current HIP device for a launch; free when it already is."""
    if dev.index is None or dev.index == torch.cuda.current_device():
        return _NO_GUARD
    return torch.cuda.device(dev)


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else C.c_void_p(t.data_ptr())


_extra_mixer_flags = 0


class mixer_flags:
    """Context manager that ORs FLARE_FLAG_* bits into every mixer descriptor built inside it (e.g.
    ``_lib.FLAG_MFMA16`` to time or test the 16x16x32 kernels where the 32x32x16 gather and scatter would run)."""

    def __init__(self, flags: int):
        self.flags = int(flags)

    def __enter__(self):
        global _extra_mixer_flags
        self.saved = _extra_mixer_flags
        _extra_mixer_flags |= self.flags
        return self

    def __exit__(self, *exc):
        global _extra_mixer_flags
        _extra_mixer_flags = self.saved
        return False


def _mixer_desc(q4, k, v, y, scale, n_splits, force_generic, drop=None) -> FlareMixerDesc:
    """drop = (p, seed) of attention dropout, or None."""
    B, H, N, D = k.shape
    d = FlareMixerDesc()
    if drop is not None:
        d.dropout_p, d.dropout_seed = float(drop[0]), int(drop[1]) & 0xFFFFFFFFFFFFFFFF
    d.B, d.H, d.N, d.M, d.D = B, H, N, q4.shape[2], D
    d.dtype = _dtype_code(k)
    d.scale = float(scale)
    d.n_splits = int(n_splits)
    d.flags = (_lib.FLAG_FORCE_GENERIC if force_generic else 0) | _extra_mixer_flags
    d.q_stride = _s3(q4)
    d.k_stride = _s3(k)
    d.v_stride = _s3(v if v is not None else k)
    d.y_stride = _s3(y if y is not None else k)
    return d


def _check_mixer_shapes(q4, k, v):
    if k.dim() != 4:
        raise ValueError(f"k must be [B,H,N,D], got {tuple(k.shape)}")
    if v is not None and v.shape != k.shape:
        raise ValueError(f"v {tuple(v.shape)} must match k {tuple(k.shape)}")
    B, H, N, D = k.shape
    if q4.shape[0] != B or q4.shape[1] != H or q4.shape[3] != D:
        raise ValueError(f"q {tuple(q4.shape)} does not match k {tuple(k.shape)}")


def _mask_u8(key_mask, B, N, device):
    if key_mask is None:
        return None
    if key_mask.shape != (B, N):
        raise ValueError(f"key_mask must be [B,N]=({B},{N}), got {tuple(key_mask.shape)}")
    return key_mask.to(device=device, dtype=torch.uint8).contiguous()


def mixer_kernel_name(q, k, v=None, scale=1.0, force_generic=False) -> str:
    """Which kernel family the dispatcher picks for these operands (no launch)."""
    r = _latent_copies(q, k, force_generic)
    if r > 1:                               # copies of every latent, see flare_multihead_mixer
        q = q.repeat(*([1] * (q.dim() - 2)), r, 1)
    M, D = q.shape[-2], k.shape[-1]
    if (M % 32 != 0 and not force_generic and q.dtype == k.dtype and D < 64 and k.dtype in (torch.bfloat16, torch.float16)
            and k.device.type == "cuda" and _dead_latent_bias(float(scale), k.dtype) is not None):
        # dead latents and a wider head, see _mixer_odd_latents
        Dp = 16 if D < 16 else 32 if D < 32 else 64
        q = q.new_zeros(*q.shape[:-2], -(-M // 32) * 32, Dp)
        k, v = _pad_last(k, Dp - D), None
    pad = _narrow_head_pad(q, k, force_generic) if q.dtype == k.dtype else 0
    if pad:                                 # what flare_multihead_mixer hands to the library for a narrow head
        q, k, v = _pad_last(q, pad), _pad_last(k, pad), None
    q4 = _q4(q, k.shape[0])
    d = _mixer_desc(q4, k, v, None, scale, 0, force_generic)
    name = _lib.load().flare_mixer_kernel_name(C.byref(d))
    if name is None:
        raise ValueError(_lib.last_error())
    return name.decode()


def _autocast_dtype(t):
    """The dtype torch.autocast would run scaled_dot_product_attention in on t's device, or None."""
    if t.device.type == "cuda" and torch.is_autocast_enabled("cuda"):
        return torch.get_autocast_dtype("cuda")
    return None


def _mixer_forward(q, k, v, scale, key_mask, n_splits, force_generic, token_major=False, want_lse=False, drop=None):
    """y, z (and with want_lse the two log-sum-exps the HIP backward needs); drop = (p, seed): attention dropout."""
    _require_cuda(q, k, v)
    lib = _lib.load()
    if q.dtype != k.dtype:
        q = q.to(k.dtype)
    if v.dtype != k.dtype:
        raise TypeError("k and v must share a dtype")
    k, v = _rows_last_contig(k), _rows_last_contig(v)
    q4 = _q4(q, k.shape[0])
    _check_mixer_shapes(q4, k, v)
    B, H, N, D = k.shape
    M = q4.shape[2]
    if token_major:   # memory order [B,N,H,D]: the head merge 'b h n d -> b n (h d)' is then a free view
        y = torch.empty((B, N, H, D), dtype=k.dtype, device=k.device).permute(0, 2, 1, 3)
    else:
        y = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    z = torch.empty((B, H, M, D), dtype=torch.float32, device=k.device)
    mask = _mask_u8(key_mask, B, N, k.device)
    d = _mixer_desc(q4, k, v, y, scale, n_splits, force_generic, drop)
    need = C.c_size_t(0)
    _lib.check(lib.flare_mixer_workspace_bytes(C.byref(d), C.byref(need)), "flare_mixer_workspace_bytes")
    ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=k.device)
    st = C.c_void_p(_stream_ptr(k.device))
    if want_lse:
        lse_lat = torch.empty((B, H, M), dtype=torch.float32, device=k.device)
        lse_tok = torch.empty((B, H, N), dtype=torch.float32, device=k.device)
        with _on_device(k.device):
            rc = lib.flare_gather_fwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(mask), _ptr(z), _ptr(lse_lat),
                                      _ptr(ws), ws.numel(), st)
            _lib.check(rc, "flare_gather_fwd")
            rc = lib.flare_scatter_fwd_lse(C.byref(d), _ptr(q4), _ptr(k), _ptr(z), _ptr(mask), _ptr(y), _ptr(lse_tok), st)
        _lib.check(rc, "flare_scatter_fwd_lse")
        return y, z, lse_lat, lse_tok
    with _on_device(k.device):
        rc = lib.flare_mixer_fwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(mask), _ptr(y), _ptr(z),
                                 _ptr(ws), ws.numel(), st)
    _lib.check(rc, "flare_mixer_fwd")
    return y, z


def _hip_backward_ok(q, k, v, key_mask, force_generic, drop=None) -> bool:
    """True when flare_mixer_bwd covers this problem (bf16/f16 and fp32, supported M, D, strides; a key mask is
    handled around the kernels, see _MixerFn.backward)."""
    if force_generic or k.dtype not in (torch.bfloat16, torch.float16, torch.float32):
        return False
    if q.dtype != k.dtype or v.dtype != k.dtype or k.device.type != "cuda":
        return False
    k, v = _rows_last_contig(k), _rows_last_contig(v)
    q4 = _q4(q, k.shape[0])
    if any(t.data_ptr() % 16 for t in (q4, k, v)):      # the kernels read 16-byte chunks: a view that starts off
        return False                                    # that grid differentiates through the torch recomputation
    d = _mixer_desc(q4, k, v, None, 1.0, 0, False, drop)
    need = C.c_size_t(0)
    return _lib.load().flare_mixer_bwd_workspace_bytes(C.byref(d), C.byref(need)) == _lib.FLARE_OK


def _mixer_hip_grad(q, k, v, y, z, lse_lat, lse_tok, scale, gy, drop=None, flags=0, dq_parts=False):
    """dq (fp32), dk, dv from the HIP backward kernels (flare_mixer_bwd); drop = (p, seed) of the forward's attention dropout.
    dq_parts (16-bit types): in dq's place (descriptor, workspace, the partial results' byte offset in it, splits)."""
    lib = _lib.load()
    k, v = _rows_last_contig(k), _rows_last_contig(v)
    B, H, N, D = k.shape
    q4 = _q4(q, B)
    M = q4.shape[2]
    gy = gy.to(k.dtype)
    per16 = 16 // k.element_size()       # elements in 16 bytes
    if gy.stride(-1) != 1 or any(s % per16 for s in gy.stride()[:3]) or gy.data_ptr() % 16:
        gy = gy.contiguous()
    d = _mixer_desc(q4, k, v, y, scale, 0, False, drop)
    d.flags |= flags
    dq = None if dq_parts else torch.empty((B, H, M, D), dtype=torch.float32, device=k.device)
    if dq_parts:
        d.flags |= _lib.FLAG_DQ_PARTS
    # k and v that are token-major views ([B,N,H,D] storage, as a projection's output is) get their gradients in the
    # same layout: the projection's backward then reads them as [B*N, H*D] rows without a copy
    like_kv = all(t.stride() == (N * H * D, D, H * D, 1) for t in (k, v)) and H > 1
    if like_kv:
        d.flags |= _lib.FLAG_GRAD_LIKE_KV
        dk = torch.empty((B, N, H, D), dtype=k.dtype, device=k.device).permute(0, 2, 1, 3)
        dv = torch.empty((B, N, H, D), dtype=k.dtype, device=k.device).permute(0, 2, 1, 3)
    else:
        dk = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
        dv = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    need = C.c_size_t(0)
    _lib.check(lib.flare_mixer_bwd_workspace_bytes(C.byref(d), C.byref(need)), "flare_mixer_bwd_workspace_bytes")
    ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=k.device)
    with _on_device(k.device):
        rc = lib.flare_mixer_bwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(y), _ptr(z), _ptr(lse_lat), _ptr(lse_tok),
                                 _ptr(gy), _s3(gy), _ptr(dq), _ptr(dk), _ptr(dv), _ptr(ws), ws.numel(),
                                 C.c_void_p(_stream_ptr(k.device)))
    _lib.check(rc, "flare_mixer_bwd")
    if dq_parts:
        off, splits = C.c_size_t(0), C.c_int32(0)
        _lib.check(lib.flare_mixer_bwd_dq_parts(C.byref(d), C.byref(off), C.byref(splits)), "flare_mixer_bwd_dq_parts")
        return (d, ws, off.value, splits.value), dk, dv
    return dq if q.dim() != 3 else dq[0] if B == 1 else dq.sum(0), dk, dv


#: elements of one [B,H,M,T] fp32 temporary of the tiled gradients below (64 MiB); about six such temporaries are
#: alive at a time, whatever N is
GRAD_TILE_ELEMS = 1 << 24


def _grad_tile(B, H, M, N) -> int:
    return int(min(N, max(256, GRAD_TILE_ELEMS // max(1, B * H * M))))


_M32 = 0xFFFFFFFF


def _lowbias32(x):
    x = x ^ (x >> 16)
    x = (x * 0x7FEB352D) & _M32
    x = x ^ (x >> 15)
    x = (x * 0x846CA68B) & _M32
    return x ^ (x >> 16)


def _p32(p: float) -> float:
    """p as the library sees it: rounded to float32 on its way through the C ABI."""
    return struct.unpack("f", struct.pack("f", p))[0]


def _dropout_threshold(p: float) -> int:
    """The 24-bit threshold the kernels compare the hash with (floor(p * 2^24) of the float32 p)."""
    return int(_p32(p) * 16777216.0)


def _dropout_keep(seed: int, phase: int, B, H, M, n0, n1, p: float, device):
    """The keep mask [B,H,M,n1-n0] of attention dropout, bit for bit the decision the kernels take
    (dropout_hash24 in csrc/common.hpp): 32-bit wrap-around arithmetic carried out in int64."""
    thr = _dropout_threshold(p)
    bh = torch.arange(B * H, device=device, dtype=torch.int64).view(B, H, 1, 1)
    m = torch.arange(M, device=device, dtype=torch.int64).view(1, 1, M, 1)
    n = torch.arange(n0, n1, device=device, dtype=torch.int64).view(1, 1, 1, -1)
    x = ((seed & _M32) + n * 0x9E3779B1 + m * 0x85EBCA77 + bh * 0xC2B2AE3D + phase * 0x27D4EB2F) & _M32
    x = _lowbias32(_lowbias32(x) ^ ((seed >> 32) & _M32))
    return (x >> 8) >= thr


def _gather_stats_tiled(qe, k, v, scale, keep, T, drop=None):
    """Log-sum-exp L [B,H,M] and z [B,H,M,D] of the gather by an online softmax over token tiles of T (fp32).
    A latent row without a single real token gets L = +inf (so that exp(s - L) = 0 below) and z = 0."""
    B, H, N, D = k.shape
    M = qe.shape[2]
    dev = k.device
    m_run = torch.full((B, H, M), float("-inf"), device=dev)
    l_run = torch.zeros((B, H, M), device=dev)
    acc = torch.zeros((B, H, M, D), device=dev) if v is not None else None
    m_safe = torch.zeros((B, H, M), device=dev)
    for n0 in range(0, N, T):
        s = scale * (qe @ k[:, :, n0:n0 + T].float().mT)
        if keep is not None:
            s = s.masked_fill(~keep[:, None, None, n0:n0 + T], float("-inf"))
        m_new = torch.maximum(m_run, s.amax(-1))
        m_safe = torch.where(torch.isfinite(m_new), m_new, torch.zeros_like(m_new))
        p = torch.exp(s - m_safe[..., None])
        alpha = torch.exp(m_run - m_safe)
        l_run = l_run * alpha + p.sum(-1)
        if acc is not None:
            if drop is not None:     # the numerator keeps the surviving weights (scaled), the denominator all of them
                p = p * _dropout_keep(drop[1], 0, B, H, M, n0, min(N, n0 + T), drop[0], dev) / (1.0 - drop[0])
            acc = acc * alpha[..., None] + p @ v[:, :, n0:n0 + T].float()
        m_run = m_new
    some = l_run > 0
    L = torch.where(some, m_safe + torch.log(l_run.clamp_min(1e-37)), torch.full_like(l_run, float("inf")))
    z = None if acc is None else torch.where(some[..., None], acc / l_run.clamp_min(1e-37)[..., None], torch.zeros_like(acc))
    return L, z


def _mixer_torch_grad(q, k, v, scale, key_mask, gy, drop=None, stats=None):
    """dq, dk, dv of the mixer by recomputation in plain torch ops on the device: used for what the HIP backward
    does not cover (fp32, unusual shapes); the forward never takes this path.  The scores are recomputed in token
    tiles of [B,H,M,T] (GRAD_TILE_ELEMS), never as the whole [B,H,M,N] matrix, with the formulas of the HIP
    backward: A = exp(S - L_m), B = exp(S - rho_n), dz = B dy, Delta = <dz,z>, delta = <dy,y>,
    dS = A (dz v^T - Delta) + B (z dy^T - delta), dv = A^T dz, dk = s dS^T q, dq = s dS k.
    drop = (p, seed): attention dropout as the forward kernels applied it; with keep masks K1, K2 (recomputed from
    the seed) and r = 1 / (1 - p) the weights that met v and z were A K1 r and B K2 r, so
    dz = (B K2 r) dy, dS = A (K1 r dz v^T - Delta) + B (K2 r z dy^T - delta), dv = (A K1 r)^T dz.
    stats = (L, z, y) as the forward's kernels left them (no mask, no dropout) spares their recomputation."""
    B, H, N, D = k.shape
    qe = (q if q.dim() == 4 else q.unsqueeze(0)).float()
    M = qe.shape[2]
    keep = None if key_mask is None else key_mask.to(torch.bool)
    T = _grad_tile(B, H, M, N)
    gy = gy if keep is None else gy * keep[:, None, :, None].to(gy.dtype)
    y = None
    if stats is not None:
        L, z, y = stats
    elif (drop is None and keep is None and k.is_cuda and q.dtype == k.dtype == v.dtype == torch.float32 and D <= 128):
        # the latents' log-sum-exp and z from the forward's own gather kernel (fp32: matrix cores) instead of a torch pass
        z, L = _gather_forward(q, k, v, scale, None, 0, False)
    else:
        L, z = _gather_stats_tiled(qe, k, v, scale, keep, T, drop)
    rs = 1.0 if drop is None else 1.0 / (1.0 - drop[0])
    # The score tiles are taken token-major, [B,H,T,M]: the softmax over the latents then runs along the last axis
    # (torch's kernel for an inner axis is an order of magnitude slower), and the products take transposed views.
    qs = scale * qe  # the scale rides on the small operand instead of a pass over every score tile
    dz = torch.zeros_like(z)
    for n0 in range(0, N, T):
        sT = k[:, :, n0:n0 + T].float() @ qs.mT
        BT = torch.softmax(sT, dim=-1)
        if drop is not None:
            BT = BT * _dropout_keep(drop[1], 1, B, H, M, n0, min(N, n0 + T), drop[0], k.device).mT * rs
        dz += BT.mT @ gy[:, :, n0:n0 + T].float()
    Delta = (dz * z).sum(-1)
    gq = torch.zeros((B, H, M, D), device=k.device)
    gk = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    gv = torch.empty((B, H, N, D), dtype=v.dtype, device=k.device)
    for n0 in range(0, N, T):
        kt, vt, gyt = k[:, :, n0:n0 + T].float(), v[:, :, n0:n0 + T].float(), gy[:, :, n0:n0 + T].float()
        sT = kt @ qs.mT
        BT = torch.softmax(sT, dim=-1)
        if keep is not None:
            sT = sT.masked_fill(~keep[:, None, n0:n0 + T, None], float("-inf"))
        AT = sT.sub_(L[:, :, None, :]).exp_()
        if drop is None:
            delta = (gyt * (BT @ z if y is None else y[:, :, n0:n0 + T].float())).sum(-1)
            dST = (vt @ dz.mT).sub_(Delta[:, :, None, :]).mul_(AT)
            dST.addcmul_(BT, (gyt @ z.mT).sub_(delta[..., None]))
        else:
            n1 = min(N, n0 + T)
            K1 = _dropout_keep(drop[1], 0, B, H, M, n0, n1, drop[0], k.device).mT * rs
            K2 = _dropout_keep(drop[1], 1, B, H, M, n0, n1, drop[0], k.device).mT * rs
            delta = (gyt * ((BT * K2) @ z)).sum(-1)
            dST = AT * (K1 * (vt @ dz.mT) - Delta[:, :, None, :]) + BT * (K2 * (gyt @ z.mT) - delta[..., None])
            AT = AT * K1
        gv[:, :, n0:n0 + T] = (AT @ dz).to(gv.dtype)
        gk[:, :, n0:n0 + T] = (dST @ qs).to(gk.dtype)
        gq += dST.mT @ kt
    gq *= scale
    if q.dim() == 3:
        gq = gq.sum(0)
    return gq.to(q.dtype), gk, gv


def _masked_hip_grad(q, k, v, y, z, lse_lat, lse_tok, scale, km, gy, drop=None):
    """_mixer_hip_grad for a problem that may carry a key mask."""
    if km is not None and drop is None:
        # The kernels know a padded token by its log-sum-exp; a batch element without a single real token has lse_lat = -inf.
        lse_tok = torch.where(km.to(torch.bool)[:, None, :], lse_tok, 2e30)
        return _mixer_hip_grad(q, k, v, y, z, torch.nan_to_num(lse_lat, nan=1e30, posinf=1e30, neginf=1e30), lse_tok, scale, gy,
                               flags=_lib.FLAG_ABSENT_TOKENS)
    if km is not None:
        # With dropout.  A padded token takes no part in either softmax.  The kernels need no mask for that: with its k, v
        # and dy rows zeroed it adds nothing to dq or dz, with its log-sum-exp set far above any score its
        # scatter weights vanish, and its own dk, dv rows are cleared afterwards.  A batch element without
        # a single real token has lse_lat = -inf; the same treatment turns its gather weights into 0.
        keep = km.to(torch.bool)
        m4 = keep[:, None, :, None]
        zero = torch.zeros((), dtype=k.dtype, device=k.device)
        k, v, gy = torch.where(m4, k, zero), torch.where(m4, v, zero), torch.where(m4, gy.to(k.dtype), zero)
        lse_tok = torch.where(keep[:, None, :], lse_tok, 1e30)
        lse_lat = torch.where(torch.isfinite(lse_lat), lse_lat, 1e30)
    gq, gk, gv = _mixer_hip_grad(q, k, v, y, z, lse_lat, lse_tok, scale, gy, drop)
    if km is not None:
        gk, gv = torch.where(m4, gk, zero), torch.where(m4, gv, zero)
    return gq, gk, gv


def _pad_rows(ts, width, token_major=None):
    """[B,H,N,D] tensors of one shape and type as [B,H,N,width], filled up with zeros or cut, in one launch; in memory [B,N,H,width] where the tensor (or
    token_major) says so, else [B,H,N,width]."""
    B, H, N, D = ts[0].shape
    if any(t.shape != ts[0].shape or t.dtype != ts[0].dtype or t.device != ts[0].device for t in ts):      # one set of sizes for the launch
        raise ValueError(f"rows to be filled up must match: {', '.join(f'{tuple(t.shape)} {t.dtype} {t.device}' for t in ts)}")
    ts = [_rows_last_contig(t) for t in ts]
    if any(s < 0 for t in ts for s in t.stride()):
        ts = [t.contiguous() for t in ts]
    out = []
    for t in ts:
        if t.stride(1) < t.stride(2) if token_major is None else token_major:
            out.append(torch.empty(B, N, H, width, dtype=t.dtype, device=t.device).permute(0, 2, 1, 3))
        else:
            out.append(torch.empty(B, H, N, width, dtype=t.dtype, device=t.device))
    if ts[0].numel() == 0:
        return [o.zero_() for o in out]
    n, k = (C.c_int64 * 3)(B, H, N), len(ts)
    with _on_device(ts[0].device):
        rc = _lib.load().flare_pad_rows(k, ts[0].element_size(), n, D, width, (C.c_void_p * k)(*(t.data_ptr() for t in ts)),
                                        (C.c_int64 * (3 * k))(*(s for t in ts for s in t.stride()[:3])), (C.c_void_p * k)(*(t.data_ptr() for t in out)),
                                        (C.c_int64 * (3 * k))(*(s for t in out for s in t.stride()[:3])), C.c_void_p(_stream_ptr(ts[0].device)))
    _lib.check(rc, "flare_pad_rows")
    return out


class _MixerFn(torch.autograd.Function):
    """q16: q as the kernels take it (cast for autocast, its heads filled up with zero columns to those of k and v), where that is
    another tensor; the gradient then goes to q itself, in q's type and width, without the cast's and the padding's own nodes.
    pad: so many columns of zeros are appended to k and v here (q16 has them), and y comes back at their width."""

    @staticmethod
    def forward(ctx, q, k, v, scale, key_mask, n_splits, force_generic, token_major, q16=None, pad=0):
        ctx.scale, ctx.key_mask = scale, key_mask
        ctx.q_dtype, ctx.q_width = q.dtype, q.shape[-1]
        ctx.set_materialize_grads(False)      # z's gradient, which nobody reads, would be a launch
        if q16 is not None:
            q = q16
        ctx.pad = pad
        if pad:
            ctx.kv_width, ctx.kv_major = k.shape[-1], tuple(t.stride(1) < t.stride(2) for t in (k, v))
            k, v = _pad_rows((k, v), k.shape[-1] + pad)
        ctx.hip = _hip_backward_ok(q, k, v, key_mask, force_generic)
        if ctx.hip:
            y, z, lse_lat, lse_tok = _mixer_forward(q, k, v, scale, key_mask, n_splits, force_generic, token_major, True)
            ctx.save_for_backward(q, k, v, y, z, lse_lat, lse_tok)
        elif (key_mask is None and k.is_cuda and q.dtype == k.dtype == v.dtype == torch.float32
              and any(t.requires_grad for t in (q, k, v))):
            # the torch recomputation starts from the latents' log-sum-exp and z: keep the forward's own
            y, z, lse_lat, _ = _mixer_forward(q, k, v, scale, None, n_splits, force_generic, token_major, True)
            ctx.save_for_backward(q, k, v, z, lse_lat, y)
        else:
            y, z = _mixer_forward(q, k, v, scale, key_mask, n_splits, force_generic, token_major)
            ctx.save_for_backward(q, k, v)
        if ctx.pad:       # token-major rows at their own width, so that merging the heads stays free; else a view
            y = _pad_rows((y,), ctx.kv_width, True)[0] if token_major else y[..., :ctx.kv_width]
            z = z[..., :ctx.kv_width]
        ctx.mark_non_differentiable(z)
        return y, z

    @staticmethod
    @once_differentiable
    def backward(ctx, gy, _gz):
        if gy is None:
            return (None,) * 10
        if ctx.pad:
            gy = _pad_rows((gy,), ctx.saved_tensors[0].shape[-1])[0]
        if ctx.hip:
            q, k, v, y, z, lse_lat, lse_tok = ctx.saved_tensors
            gq, gk, gv = _masked_hip_grad(q, k, v, y, z, lse_lat, lse_tok, ctx.scale, ctx.key_mask, gy)
        else:
            q, k, v, *stats = ctx.saved_tensors
            gq, gk, gv = _mixer_torch_grad(q, k, v, ctx.scale, ctx.key_mask, gy,
                                           stats=(stats[1], stats[0], stats[2]) if stats else None)
        if ctx.pad:
            gk, gv = (_pad_rows((gk, gv), ctx.kv_width, ctx.kv_major[0]) if ctx.kv_major[0] == ctx.kv_major[1] else
                      [_pad_rows((t,), ctx.kv_width, m)[0] for t, m in zip((gk, gv), ctx.kv_major)])
        return gq[..., :ctx.q_width].to(ctx.q_dtype), gk, gv, None, None, None, None, None, None, None


def mixer_narrow_heads(q, k, v, scale):
    """y of the differentiable mixer for latents q [H,M,D] and 16-bit k, v [B,H,N,16] whose heads hold D channels followed by zeros (as
    the projections write them); y is head-padded like them, token-major in memory."""
    q16 = torch.zeros(*q.shape[:-1], k.shape[-1], dtype=k.dtype, device=k.device)
    with torch.no_grad():
        q16[..., :q.shape[-1]].copy_(q)
    return _MixerFn.apply(q, k, v, float(scale), None, 0, False, True, q16)[0]


class _MixerDropoutFn(torch.autograd.Function):
    """The mixer with attention dropout.  Where flare_mixer_bwd takes the problem (fp32 on the matrix cores) the backward
    runs there and regenerates the keep masks from (p, seed); elsewhere it is the tiled torch recomputation with the
    same masks (_dropout_keep)."""

    @staticmethod
    def forward(ctx, q, k, v, scale, key_mask, p, seed, token_major):
        ctx.scale, ctx.key_mask, ctx.drop = scale, key_mask, (p, seed)
        ctx.hip = _hip_backward_ok(q, k, v, key_mask, False, ctx.drop)
        if ctx.hip:
            y, z, lse_lat, lse_tok = _mixer_forward(q, k, v, scale, key_mask, 0, False, token_major, True, ctx.drop)
            ctx.save_for_backward(q, k, v, y, z, lse_lat, lse_tok)
        else:
            y, z = _mixer_forward(q, k, v, scale, key_mask, 0, False, token_major, False, ctx.drop)
            ctx.save_for_backward(q, k, v)
        ctx.mark_non_differentiable(z)
        return y, z

    @staticmethod
    @once_differentiable
    def backward(ctx, gy, _gz):
        if ctx.hip:
            q, k, v, y, z, lse_lat, lse_tok = ctx.saved_tensors
            gq, gk, gv = _masked_hip_grad(q, k, v, y, z, lse_lat, lse_tok, ctx.scale, ctx.key_mask, gy, ctx.drop)
            gq = gq.to(q.dtype)
        else:
            q, k, v = ctx.saved_tensors
            gq, gk, gv = _mixer_torch_grad(q, k, v, ctx.scale, ctx.key_mask, gy, ctx.drop)
        return gq, gk, gv, None, None, None, None, None


def _narrow_head_pad(q, k, force_generic) -> int:
    """Columns of zeros to append to a head dim so that the matrix-core kernels (D in {16, 32, 64}) take the problem,
    or 0.  Zero columns change neither the scores q.k nor the first D output columns; the reference's default model
    has D = channel_dim / num_heads = 8, which the fp32-FMA kernels would serve 5-15x slower.  fp32 problems have
    matrix-core kernels too (latent counts that are multiples of 16)."""
    D = k.shape[-1]
    if force_generic or D > 64 or k.device.type != "cuda":
        return 0
    target = 16 if D <= 16 else 32 if D <= 32 else 64
    if k.dtype == torch.float32:
        return target - D if q.shape[-2] % 16 == 0 else 0
    if k.dtype not in (torch.bfloat16, torch.float16):
        return 0
    return target - D if q.shape[-2] % 32 == 0 else 0


def _pad_last(t, n):
    return torch.nn.functional.pad(t, (0, n))


def flare_multihead_mixer(q, k, v, scale: float = 1.0, key_mask=None, return_z: bool = False,
                          n_splits: int = 0, force_generic: bool = False, token_major_out: bool = False,
                          dropout_p: float = 0.0, dropout_seed: Optional[int] = None):
    """FLARE gather-scatter mixer (README.md:39-52 of the reference).

    q: [H,M,D] latent queries (or [B,H,M,D]); k, v: [B,H,N,D]; returns y [B,H,N,D] with
      z = softmax_n(scale q k^T) v ;  y = softmax_m(scale k q^T) z
    key_mask ([B,N], nonzero = token present) removes padded tokens from the gather and
    zeroes their output rows (lra/models/backends.py:603-606,615-622).
    k and v may be strided views (e.g. 'b n (h d) -> b h n d') as long as D is contiguous.
    Under torch.autocast the operands are cast to the autocast dtype, as torch does for the
    scaled_dot_product_attention calls this replaces.  token_major_out=True lays y out as
    [B,N,H,D] in memory (returned as its [B,H,N,D] view) so that merging the heads is free.
    dropout_p > 0 drops entries of both softmaxes' weights the way torch's scaled_dot_product_attention does
    in training (lra/models/backends.py:592,605-606); the mask is a function of dropout_seed (drawn from torch's
    default generator when None), so the backward recomputes it.  The 32x32x16 kernels carry no dropout: 16-bit problems
    run forward and backward on the 16x16x32 kernels, fp32 problems on the fp32 matrix-core kernels.
    """
    ac = _autocast_dtype(k)
    q_in = q
    if ac is not None:
        q, k, v = (t if t.dtype == ac else t.to(ac) for t in (q, k, v))
    q_cast = q
    if dropout_p > 0.0:
        if not dropout_p < 1.0:
            raise ValueError("dropout_p must be in [0, 1)")
        seed = int(torch.randint(0, 2 ** 62, (), dtype=torch.int64)) if dropout_seed is None else int(dropout_seed)
        D = k.shape[-1]
        # zero columns change neither the scores nor the mask's indices: narrow heads reach the matrix-core kernels
        pad = _narrow_head_pad(q, k, force_generic) if q.dtype == k.dtype == v.dtype else 0
        if pad:
            q, k, v = _pad_last(q, pad), _pad_last(k, pad), _pad_last(v, pad)
        if torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v)):
            y, z = _MixerDropoutFn.apply(q, k, v, float(scale), key_mask, float(dropout_p), seed, token_major_out)
        else:
            y, z = _mixer_forward(q, k, v, float(scale), key_mask, 0, force_generic, token_major_out, False,
                                  (float(dropout_p), seed))
        if pad:
            y, z = y[..., :D], z[..., :D]
        return (y, z) if return_z else y
    D = k.shape[-1]
    r = _latent_copies(q, k, force_generic)
    if r > 1 and q.dtype == v.dtype:
        # r copies of every latent: each copy gathers the same row of z and the softmax over the r*M copies gives each
        # 1/r of the weight latent m had, so y is unchanged; autograd sums the copies' gradients through repeat()
        M = q.shape[-2]
        out = flare_multihead_mixer(q.repeat(*([1] * (q.dim() - 2)), r, 1), k, v, scale, key_mask, return_z, n_splits,
                                    force_generic, token_major_out)
        return (out[0], out[1][..., :M, :]) if return_z else out
    if (q.shape[-2] % 32 != 0 and not force_generic and q.dtype == k.dtype == v.dtype and D < 64
            and k.dtype in (torch.bfloat16, torch.float16) and k.device.type == "cuda"
            and _dead_latent_bias(float(scale), k.dtype) is not None):
        return _mixer_odd_latents(q, k, v, float(scale), key_mask, return_z, n_splits, token_major_out)
    pad = _narrow_head_pad(q, k, force_generic) if q.dtype == k.dtype == v.dtype else 0
    needs_grad = torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v))
    if pad and not (k.dim() == v.dim() == 4 and k.shape == v.shape and q.device == k.device == v.device):
        q, k, v, pad = _pad_last(q, pad), _pad_last(k, pad), _pad_last(v, pad), 0      # refused below
    if needs_grad and return_z:
        # z is handed out and may enter a loss of its own: take the two differentiable halves, so that gradients
        # reach q, k, v through z as well as through y (the fused function below treats z as an internal value)
        if pad:
            q, k, v = _pad_last(q, pad), _pad_last(k, pad), _pad_last(v, pad)
        z, _ = flare_gather(q, k, v, scale, key_mask, n_splits, force_generic)
        y = flare_scatter(q, k, z, scale, key_mask, force_generic)
        if token_major_out:
            y = y.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    elif needs_grad:
        # the cast of the latents for autocast, and zero columns for narrow heads, stay inside the function
        cast = q is q_cast and q is not q_in and q_in.dtype == torch.float32
        q16 = _pad_last(q.detach(), pad) if pad else q.detach() if cast else None
        y, z = _MixerFn.apply(q_in if cast else q, k, v, float(scale), key_mask, n_splits, force_generic, token_major_out, q16, pad)
        return (y, z) if return_z else y
    else:
        if pad:
            q, (k, v) = _pad_last(q, pad), _pad_rows((k, v), D + pad)
        y, z = _mixer_forward(q, k, v, float(scale), key_mask, n_splits, force_generic, token_major_out)
    if pad:
        y, z = y[..., :D], z[..., :D]
    return (y, z) if return_z else y


def _latent_copies(q, k, force_generic) -> int:
    """How many copies of every latent bring a 16-bit problem's latent count to a multiple of 32 (what the matrix-core
    kernels and the HIP backward take): 2 or 4 for multiples of 8, else 1 (other counts get dead latents instead)."""
    M, D = q.shape[-2], k.shape[-1]
    if (M % 32 == 0 or M % 8 != 0 or force_generic or D > 64 or q.dtype != k.dtype
            or k.dtype not in (torch.bfloat16, torch.float16) or k.device.type != "cuda"):
        return 1
    return 32 // math.gcd(M, 32)


def _dead_latent_bias(scale: float, dtype):
    """The entry a dead latent's query holds in the column of ones (see _mixer_odd_latents): its score is
    scale * bias, which has to sit at least 200 below any real score's neighbourhood whatever the scale is.
    None when the element type cannot hold such a value (f16 with a scale below about 200 / 60000)."""
    if not scale > 0.0:
        return None
    need = max(16384.0, 256.0 / scale)        # 256 rather than 200: room for the rounding to the element type
    limit = 60000.0 if dtype == torch.float16 else 1.0e30
    return -need if need <= limit else None


def _mixer_odd_latents(q, k, v, scale, key_mask, return_z, n_splits, token_major_out):
    """A latent count that is not a multiple of 32 on the matrix-core kernels: the latents are filled up with dead
    ones.  In the gather a dead latent is a zero query whose row of z is never used.  In the scatter it must get no
    weight: k receives one extra column of ones and the dead queries hold a large negative number there (the real
    ones 0; -16384, or -256 / scale when the scale is small, so that scale * bias stays below -200), which takes
    their scores out of every token's softmax.  The extra column rides in the zero padding of the head dim (D grows to
    the next of 16, 32, 64 that leaves room for it).  Gradients come from the two halves' own backward."""
    M, D = q.shape[-2], k.shape[-1]
    Mp = -(-M // 32) * 32
    Dp = 16 if D < 16 else 32 if D < 32 else 64
    qz = _pad_last(q, Dp - D)
    dead = qz.new_zeros(*qz.shape[:-2], Mp - M, Dp)
    q_gather = torch.cat([qz, dead], dim=-2)
    dead_s = dead.clone()
    dead_s[..., D] = _dead_latent_bias(scale, k.dtype)
    q_scatter = torch.cat([qz, dead_s], dim=-2)
    kp = _pad_last(k, Dp - D).clone() if Dp - D else k
    kp[..., D] = 1.0
    vp = _pad_last(v, Dp - D)
    z, _ = flare_gather(q_gather, kp, vp, scale, key_mask, n_splits)
    y = flare_scatter(q_scatter, kp, z, scale, key_mask)
    y = y[..., :D]
    if token_major_out:
        y = y.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    return (y, z[..., :M, :D]) if return_z else y


def _gather_forward(q, k, v, scale, key_mask, n_splits, force_generic):
    _require_cuda(q, k, v)
    lib = _lib.load()
    if q.dtype != k.dtype:
        q = q.to(k.dtype)
    k, v = _rows_last_contig(k), _rows_last_contig(v)
    q4 = _q4(q, k.shape[0])
    _check_mixer_shapes(q4, k, v)
    B, H, N, D = k.shape
    M = q4.shape[2]
    z = torch.empty((B, H, M, D), dtype=torch.float32, device=k.device)
    lse = torch.empty((B, H, M), dtype=torch.float32, device=k.device)
    mask = _mask_u8(key_mask, B, N, k.device)
    d = _mixer_desc(q4, k, v, None, scale, n_splits, force_generic)
    need = C.c_size_t(0)
    _lib.check(lib.flare_mixer_workspace_bytes(C.byref(d), C.byref(need)), "flare_mixer_workspace_bytes")
    ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=k.device)
    with _on_device(k.device):
        rc = lib.flare_gather_fwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(mask), _ptr(z), _ptr(lse),
                                  _ptr(ws), ws.numel(), C.c_void_p(_stream_ptr(k.device)))
    _lib.check(rc, "flare_gather_fwd")
    return z, lse


def _scatter_forward(q, k, z, scale, key_mask, force_generic, want_lse=False):
    """y (and with want_lse each token's log-sum-exp over the latents, which the HIP backward of the half needs)."""
    _require_cuda(q, k, z)
    lib = _lib.load()
    if q.dtype != k.dtype:
        q = q.to(k.dtype)
    k = _rows_last_contig(k)
    q4 = _q4(q, k.shape[0])
    _check_mixer_shapes(q4, k, None)
    B, H, N, D = k.shape
    M = q4.shape[2]
    if z.shape != (B, H, M, D):
        raise ValueError(f"z must be [B,H,M,D]=({B},{H},{M},{D}), got {tuple(z.shape)}")
    z = z.to(torch.float32).contiguous()
    y = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    mask = _mask_u8(key_mask, B, N, k.device)
    d = _mixer_desc(q4, k, None, y, scale, 0, force_generic)
    if want_lse:
        lse_tok = torch.empty((B, H, N), dtype=torch.float32, device=k.device)
        with _on_device(k.device):
            rc = lib.flare_scatter_fwd_lse(C.byref(d), _ptr(q4), _ptr(k), _ptr(z), _ptr(mask), _ptr(y), _ptr(lse_tok),
                                           C.c_void_p(_stream_ptr(k.device)))
        _lib.check(rc, "flare_scatter_fwd_lse")
        return y, lse_tok
    with _on_device(k.device):
        rc = lib.flare_scatter_fwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(z), _ptr(mask), _ptr(y),
                                   C.c_void_p(_stream_ptr(k.device)))
    _lib.check(rc, "flare_scatter_fwd")
    return y


def _half_torch_grad(which, q, k, x, scale, key_mask, g):
    """Gradients of one half of the mixer by recomputation in plain torch ops on the device (the forward
    never takes this path), in token tiles like _mixer_torch_grad: which='gather' -> z = softmax_n(s q k^T) x with
    x = v and g = dz; which='scatter' -> y = softmax_m(s k q^T) x with x = z and g = dy."""
    B, H, N, D = k.shape
    qe = (q if q.dim() == 4 else q.unsqueeze(0)).float()
    M = qe.shape[2]
    keep = None if key_mask is None else key_mask.to(torch.bool)
    T = _grad_tile(B, H, M, N)
    gq = torch.zeros((B, H, M, D), device=k.device)
    gk = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    if which == "gather":
        L, z = _gather_stats_tiled(qe, k, x, scale, keep, T)
        dz = g.float()
        Delta = (dz * z).sum(-1)
        gx = torch.empty((B, H, N, D), dtype=x.dtype, device=k.device)
        for n0 in range(0, N, T):
            kt, vt = k[:, :, n0:n0 + T].float(), x[:, :, n0:n0 + T].float()
            s = scale * (qe @ kt.mT)
            if keep is not None:
                s = s.masked_fill(~keep[:, None, None, n0:n0 + T], float("-inf"))
            A = torch.exp(s - L[..., None])
            dS = A * (dz @ vt.mT - Delta[..., None])
            gx[:, :, n0:n0 + T] = (A.mT @ dz).to(gx.dtype)
            gk[:, :, n0:n0 + T] = (scale * (dS.mT @ qe)).to(gk.dtype)
            gq += scale * (dS @ kt)
    else:
        z = x.float()
        gy = g if keep is None else g * keep[:, None, :, None].to(g.dtype)
        gz = torch.zeros((B, H, M, D), device=k.device)
        for n0 in range(0, N, T):
            kt, gyt = k[:, :, n0:n0 + T].float(), gy[:, :, n0:n0 + T].float()
            BT = torch.softmax(scale * (kt @ qe.mT), dim=-1)       # token-major tile: the softmax runs along the last axis
            delta = (gyt * (BT @ z)).sum(-1)
            dST = BT * (gyt @ z.mT - delta[..., None])
            gz += BT.mT @ gyt
            gk[:, :, n0:n0 + T] = (scale * (dST @ qe)).to(gk.dtype)
            gq += scale * (dST.mT @ kt)
        gx = gz.to(x.dtype)
    if q.dim() == 3:
        gq = gq.sum(0)
    return gq.to(q.dtype), gk, gx


def _half_hip_ok(q, k, other, key_mask, force_generic) -> bool:
    """True when the HIP backward of a half (flare_gather_bwd / flare_scatter_bwd) covers the problem: q and k of one
    dtype, `other` (v of the gather, z of the scatter) of that dtype or, for z, fp32."""
    if force_generic or q.dtype != k.dtype or other.dtype not in (k.dtype, torch.float32) or not k.is_cuda:
        return False
    if k.dtype not in (torch.float32, torch.bfloat16, torch.float16):
        return False
    k = _rows_last_contig(k)
    q4 = _q4(q, k.shape[0])
    if any(t.data_ptr() % 16 for t in (q4, k)):
        return False
    d = _mixer_desc(q4, k, k, None, 1.0, 0, False)
    need = C.c_size_t(0)
    return _lib.load().flare_mixer_bwd_workspace_bytes(C.byref(d), C.byref(need)) == _lib.FLARE_OK


def _half_hip_grad(which, q, k, x, z, aux, scale, key_mask, g):
    """Gradients of a half from the HIP kernels.  gather: x = v, aux = lse_lat, g = dz -> (dq, dk, dv);
    scatter: x = y, aux = lse_tok, g = dy -> (dq, dk, dz).  A key mask is handled as in _MixerFn.backward."""
    lib = _lib.load()
    k = _rows_last_contig(k)
    B, H, N, D = k.shape
    q4 = _q4(q, B)
    M = q4.shape[2]
    al = 4 if k.dtype == torch.float32 else 8          # strides in elements that keep rows 16-byte aligned
    keep = None
    if key_mask is not None:
        keep = key_mask.to(torch.bool)
        m4 = keep[:, None, :, None]
        k = torch.where(m4, k, k.new_zeros(()))
    z32 = z.to(torch.float32).contiguous()
    dq = torch.empty((B, H, M, D), dtype=torch.float32, device=k.device)
    dk = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    if which == "gather":
        v = _rows_last_contig(x)
        aux = aux.contiguous()
        if keep is not None:
            v = torch.where(m4, v, v.new_zeros(()))
            aux = torch.where(torch.isfinite(aux), aux, 1e30)
        if v.data_ptr() % 16 or any(s % al for s in v.stride()[:3]):
            v = v.contiguous()
        gz = g.to(torch.float32).contiguous()
        d = _mixer_desc(q4, k, v, None, scale, 0, False)
        if keep is not None:
            d.flags |= _lib.FLAG_ABSENT_TOKENS
        out = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    else:
        y = x.contiguous()
        gy = g.to(k.dtype)
        aux = aux.contiguous()
        if keep is not None:
            gy = torch.where(m4, gy, gy.new_zeros(()))
            aux = torch.where(keep[:, None, :], aux, 1e30)
        if gy.stride(-1) != 1 or any(s % al for s in gy.stride()[:3]) or gy.data_ptr() % 16:
            gy = gy.contiguous()
        d = _mixer_desc(q4, k, k, y, scale, 0, False)
        out = torch.empty((B, H, M, D), dtype=torch.float32, device=k.device)
    need = C.c_size_t(0)
    _lib.check(lib.flare_mixer_bwd_workspace_bytes(C.byref(d), C.byref(need)), "flare_mixer_bwd_workspace_bytes")
    ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=k.device)
    st = C.c_void_p(_stream_ptr(k.device))
    with _on_device(k.device):
        if which == "gather":
            rc = lib.flare_gather_bwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(z32), _ptr(aux), _ptr(gz), _ptr(dq), _ptr(dk),
                                      _ptr(out), _ptr(ws), ws.numel(), st)
        else:
            rc = lib.flare_scatter_bwd(C.byref(d), _ptr(q4), _ptr(k), _ptr(z32), _ptr(y), _ptr(aux), _ptr(gy), _s3(gy), _ptr(dq),
                                       _ptr(dk), _ptr(out), _ptr(ws), ws.numel(), st)
    _lib.check(rc, "flare_gather_bwd" if which == "gather" else "flare_scatter_bwd")
    if keep is not None:
        dk = torch.where(m4, dk, dk.new_zeros(()))
        if which == "gather":
            out = torch.where(m4, out, out.new_zeros(()))
    if which == "scatter":
        out = out.to(z.dtype)
    gq = dq.sum(0) if q.dim() == 3 else dq
    return gq.to(q.dtype), dk, out


class _GatherFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, scale, key_mask, n_splits, force_generic):
        ctx.scale, ctx.key_mask = scale, key_mask
        z, lse = _gather_forward(q, k, v, scale, key_mask, n_splits, force_generic)
        ctx.hip = _half_hip_ok(q, k, v, key_mask, force_generic)
        if ctx.hip:
            ctx.save_for_backward(q, k, v, z, lse)
        else:
            ctx.save_for_backward(q, k, v)
        ctx.mark_non_differentiable(lse)
        return z, lse

    @staticmethod
    @once_differentiable
    def backward(ctx, gz, _glse):
        if ctx.hip:
            q, k, v, z, lse = ctx.saved_tensors
            return (*_half_hip_grad("gather", q, k, v, z, lse, ctx.scale, ctx.key_mask, gz), None, None, None, None)
        q, k, v = ctx.saved_tensors
        return (*_half_torch_grad("gather", q, k, v, ctx.scale, ctx.key_mask, gz), None, None, None, None)


class _ScatterFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, z, scale, key_mask, force_generic):
        ctx.scale, ctx.key_mask = scale, key_mask
        ctx.hip = _half_hip_ok(q, k, z, key_mask, force_generic)
        if ctx.hip:
            y, lse_tok = _scatter_forward(q, k, z, scale, key_mask, force_generic, want_lse=True)
            ctx.save_for_backward(q, k, z, y, lse_tok)
            return y
        ctx.save_for_backward(q, k, z)
        return _scatter_forward(q, k, z, scale, key_mask, force_generic)

    @staticmethod
    @once_differentiable
    def backward(ctx, gy):
        if ctx.hip:
            q, k, z, y, lse_tok = ctx.saved_tensors
            return (*_half_hip_grad("scatter", q, k, y, z, lse_tok, ctx.scale, ctx.key_mask, gy), None, None, None)
        q, k, z = ctx.saved_tensors
        return (*_half_torch_grad("scatter", q, k, z, ctx.scale, ctx.key_mask, gy), None, None, None)


def flare_gather(q, k, v, scale: float = 1.0, key_mask=None, n_splits: int = 0,
                 force_generic: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """z [B,H,M,D] fp32 = softmax_n(scale q k^T) v and lse [B,H,M] (natural log).
    Differentiable in q, k, v (flare_gather_bwd where the HIP backward covers the shape, otherwise a recomputation of the
    scores with torch ops): for models that put layers between the two halves; the whole mixer has its own backward."""
    D = k.shape[-1]
    pad = _narrow_head_pad(q, k, force_generic) if q.dtype == k.dtype == v.dtype else 0
    if pad:
        q, k, v = _pad_last(q, pad), _pad_last(k, pad), _pad_last(v, pad)
    if torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v)):
        z, lse = _GatherFn.apply(q, k, v, float(scale), key_mask, n_splits, force_generic)
    else:
        z, lse = _gather_forward(q, k, v, float(scale), key_mask, n_splits, force_generic)
    return (z[..., :D] if pad else z), lse


def flare_scatter(q, k, z, scale: float = 1.0, key_mask=None, force_generic: bool = False) -> torch.Tensor:
    """y [B,H,N,D] = softmax_m(scale k q^T) z with z [B,H,M,D] (computed from its fp32 copy).
    Differentiable in q, k, z like flare_gather."""
    D = k.shape[-1]
    pad = _narrow_head_pad(q, k, force_generic) if q.dtype == k.dtype else 0
    if pad:
        q, k, z = _pad_last(q, pad), _pad_last(k, pad), _pad_last(z, pad)
    if torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, z)):
        y = _ScatterFn.apply(q, k, z, float(scale), key_mask, force_generic)
    else:
        y = _scatter_forward(q, k, z, float(scale), key_mask, force_generic)
    return y[..., :D] if pad else y


# --------------------------------------------------------------------------------------
# causal FLARE
# --------------------------------------------------------------------------------------
def causal_fresh_state(B, H, M, D, device):
    """(mu, den, num) of an empty prefix: mu = -inf, den = 0, num = 0 (fp32)."""
    mu = torch.full((B, H, M), float("-inf"), dtype=torch.float32, device=device)
    den = torch.zeros((B, H, M), dtype=torch.float32, device=device)
    num = torch.zeros((B, H, M, D), dtype=torch.float32, device=device)
    return mu, den, num


def _causal_latent_groups(M, D):
    """Sizes of the latent groups a 16-bit causal problem is run in when the matrix-core kernels do not take its M
    in one piece: 256 (heads up to 32) or 128 latents, then powers of two down to 32 for the rest.  [] when M is not
    a multiple of 32 or D is above 64; a single entry when no split is needed."""
    if M % 32 != 0 or D > 64 or M <= 128 and M & (M - 1) == 0:
        return [M] if M % 32 == 0 and D <= 64 else []
    big = 256 if D <= 32 else 128
    sizes = [big] * (M // big)
    rest = M % big
    for p in (128, 64, 32):
        if rest >= p:
            sizes.append(p)
            rest -= p
    return sizes


#: decode calls of at least this many tokens also take the replicated-latent route below (a shorter decode is
#: launch-bound, and the fp32 step kernel reads a state half the size or less)
CAUSAL_REPLICATE_DECODE_MIN_TOKENS = 32


def _causal_join(ys, lses):
    """y = sum_g softmax_g(lse_g) y_g in one launch (flare_causal_join)."""
    lib = _lib.load()
    if ys[0].shape[-1] % 8 != 0 or len(ys) > 16:      # rows the join kernel's 16-byte accesses do not fit
        w = torch.softmax(torch.stack(lses), dim=0).unsqueeze(-1)
        return (w * torch.stack([t.float() for t in ys])).sum(0).to(ys[0].dtype)
    ys = [t.contiguous() for t in ys]
    lses = [t.contiguous() for t in lses]
    y = torch.empty_like(ys[0])
    G = len(ys)
    yp = (C.c_void_p * G)(*[t.data_ptr() for t in ys])
    lp = (C.c_void_p * G)(*[t.data_ptr() for t in lses])
    rows = y.numel() // y.shape[-1]
    with _on_device(y.device):
        rc = lib.flare_causal_join(_dtype_code(y), G, rows, y.shape[-1], yp, lp, _ptr(y), C.c_void_p(_stream_ptr(y.device)))
    _lib.check(rc, "flare_causal_join")
    return y


def _causal_call(entry, q, k, v, scale, chunk, state, want_lse=False, inplace=False, workspace=None, out=None):
    """(y, state) or, with want_lse, (y, state, lse) where lse [B,H,N] is each token's log-sum-exp over the latents."""
    _require_cuda(q, k, v)
    D = k.shape[-1]
    M = q.shape[-2]
    if (k.dtype in (torch.bfloat16, torch.float16) and M < 128 and 128 % M == 0 and D <= 64
            and q.shape[-1] == D and v.shape == k.shape and k.dim() == 4
            and (entry == "prefill" or k.shape[2] >= CAUSAL_REPLICATE_DECODE_MIN_TOKENS)):
        # The matrix-core causal kernels take 128 or 256 latents.  r copies of every latent leave y unchanged: each
        # copy carries the same running state z_m(t), and the softmax over the r*M copies gives each 1/r of the
        # weight latent m had.  So a power-of-two latent count below 128 is tiled up to 128 (state in and out
        # likewise) instead of taking the fp32 kernel.
        if inplace:
            raise ValueError("inplace=True needs a latent count the kernels take as it is (this one runs as copies)")
        r = 128 // M
        qr = q.repeat(*([1] * (q.dim() - 2)), r, 1)
        if state is not None:
            mu, den, num = state
            state = (mu.repeat(1, 1, r), den.repeat(1, 1, r), num.repeat(1, 1, r, 1))
        res = _causal_call(entry, qr, k, v, scale, chunk, state, want_lse=want_lse)
        mu, den, num = res[1]
        st = (mu[..., :M].contiguous(), den[..., :M].contiguous(), num[..., :M, :].contiguous())
        # the r copies of every latent multiply each token's softmax sum by r
        return (res[0], st, res[2] - math.log(r)) if want_lse else (res[0], st)
    groups = _causal_latent_groups(M, D) if k.dtype in (torch.bfloat16, torch.float16) else []
    if len(groups) > 1 and q.shape[-1] == D and v.shape == k.shape and k.dim() == 4:
        # A latent count the matrix-core kernels do not take in one piece (256 latents with a head above 32 exceed a
        # workgroup's LDS; 96, 192, 384, 512 ... have no kernel instance).  The softmax over the latents splits: each
        # group of latents is a causal problem of its own whose y_g is normalised within the group, and
        # y = sum_g w_g y_g with w_g = S_g / sum_g' S_g', S_g(t) = sum over the group of exp(scale <k_t, q_m>);
        # the state is per latent and is cut and joined along M.
        if inplace:
            raise ValueError("inplace=True needs a latent count the kernels take in one piece (this one runs in groups)")
        ys, sts, lses, m0 = [], [], [], 0
        for g in groups:
            sl = slice(m0, m0 + g)
            m0 += g
            st_g = None if state is None else (state[0][..., sl], state[1][..., sl], state[2][..., sl, :])
            y_g, st_g, lse_g = _causal_call(entry, q[..., sl, :], k, v, scale, chunk, st_g, want_lse=True)
            ys.append(y_g)
            sts.append(st_g)
            lses.append(lse_g)
        y = _causal_join(ys, lses)
        st = tuple(torch.cat(parts, dim=2) for parts in zip(*sts))
        if want_lse:
            return y, st, torch.logsumexp(torch.stack(lses), dim=0)
        return y, st
    if (k.dtype in (torch.bfloat16, torch.float16) and (D < 32 and M in (128, 256) or 32 < D < 64 and M == 128)
            and q.shape[-1] == D and v.shape == k.shape):
        # the matrix-core causal kernels take D = 32 and 64: any other head up to 64 gets zero columns (scores and the
        # first D columns of every output and of the state's numerators are unchanged) instead of the fp32 kernel
        if inplace:
            raise ValueError("inplace=True needs a head dim the kernels take as it is (this one is zero-padded)")
        pad = (32 if D < 32 else 64) - D
        if state is not None:
            state = (state[0], state[1], _pad_last(state[2], pad))
        res = _causal_call_launch(entry, _pad_last(q, pad), _pad_last(k, pad), _pad_last(v, pad), scale, chunk, state, want_lse)
        mu, den, num = res[1]
        st = (mu, den, num[..., :D].contiguous())
        return (res[0][..., :D], st, res[2]) if want_lse else (res[0][..., :D], st)
    return _causal_call_launch(entry, q, k, v, scale, chunk, state, want_lse, inplace, workspace, out)


def causal_workspace(q, k) -> torch.Tensor:
    """A workspace for flare_causal_* calls on operands of these shapes (for callers that reuse one across calls,
    e.g. a decode loop with inplace=True)."""
    B, H, N, D = k.shape
    y = torch.empty(0, dtype=k.dtype, device=k.device)
    d = FlareCausalDesc()
    d.B, d.H, d.N, d.M, d.D = B, H, N, q.shape[-2], D
    d.dtype = _dtype_code(k)
    d.scale = 1.0
    q4 = _q4(q, B)
    d.q_stride, d.k_stride, d.v_stride = _s3(q4), _s3(k), _s3(k)
    d.y_stride = _lib.I3(H * N * D, N * D, D)
    need = C.c_size_t(0)
    _lib.check(_lib.load().flare_causal_workspace_bytes(C.byref(d), C.byref(need)), "flare_causal_workspace_bytes")
    return torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=k.device)


def _causal_call_launch(entry, q, k, v, scale, chunk, state, want_lse=False, inplace=False, workspace=None, out=None):
    lib = _lib.load()
    if q.dtype != k.dtype:
        q = q.to(k.dtype)
    if v.dtype != k.dtype or v.shape != k.shape or k.dim() != 4:
        raise ValueError("k and v must be [B,H,N,D] tensors of one dtype")
    k, v = _rows_last_contig(k), _rows_last_contig(v)
    B, H, N, D = k.shape
    q4 = _q4(q, B)
    _check_mixer_shapes(q4, k, v)
    M = q4.shape[2]
    if state is None:
        # fresh: mu = -inf marks every latent as empty, and no kernel reads the sums of an empty latent, so den and
        # num need no fill (every element of the returned state is written by the call)
        mu = torch.full((B, H, M), float("-inf"), dtype=torch.float32, device=k.device)
        den = torch.empty((B, H, M), dtype=torch.float32, device=k.device)
        num = torch.empty((B, H, M, D), dtype=torch.float32, device=k.device)
    elif inplace:
        mu, den, num = state
        for s_ in (mu, den, num):
            if s_.dtype != torch.float32 or s_.device != k.device or not s_.is_contiguous():
                raise ValueError("inplace=True advances the given state tensors: they must be contiguous fp32 tensors on k's device")
    else:
        mu, den, num = (s.to(device=k.device, dtype=torch.float32).contiguous().clone() for s in state)
    if mu.shape != (B, H, M) or den.shape != (B, H, M) or num.shape != (B, H, M, D):
        raise ValueError("state must be (mu[B,H,M], den[B,H,M], num[B,H,M,D])")
    if out is None:
        y = torch.empty((B, H, N, D), dtype=k.dtype, device=k.device)
    else:
        y = out
        if y.shape != (B, H, N, D) or y.dtype != k.dtype or y.device != k.device or y.stride(-1) != 1:
            raise ValueError("out must be a [B,H,N,D] tensor of k's dtype and device with contiguous rows")
    lse = torch.empty((B, H, N), dtype=torch.float32, device=k.device) if want_lse else None
    d = FlareCausalDesc()
    d.B, d.H, d.N, d.M, d.D = B, H, N, M, D
    d.dtype = _dtype_code(k)
    d.scale = float(scale)
    d.chunk = int(chunk)
    d.q_stride, d.k_stride, d.v_stride, d.y_stride = _s3(q4), _s3(k), _s3(v), _s3(y)
    st = C.c_void_p(_stream_ptr(k.device))
    with _on_device(k.device):
        if workspace is None:
            need = C.c_size_t(0)
            _lib.check(lib.flare_causal_workspace_bytes(C.byref(d), C.byref(need)), "flare_causal_workspace_bytes")
            ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=k.device)
        else:
            ws = workspace          # the library checks its size and alignment
        if want_lse:
            fn = lib.flare_causal_prefill_fwd_lse if entry == "prefill" else lib.flare_causal_decode_fwd_lse
            rc = fn(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(y), _ptr(lse), _ptr(mu), _ptr(den), _ptr(num), _ptr(ws),
                    ws.numel(), st)
        else:
            fn = lib.flare_causal_prefill_fwd if entry == "prefill" else lib.flare_causal_decode_fwd
            rc = fn(C.byref(d), _ptr(q4), _ptr(k), _ptr(v), _ptr(y), _ptr(mu), _ptr(den), _ptr(num), _ptr(ws),
                    ws.numel(), st)
    _lib.check(rc, f"flare_causal_{entry}_fwd")
    return (y, (mu, den, num), lse) if want_lse else (y, (mu, den, num))


def flare_causal_prefill(q, k, v, scale: float = 1.0, chunk: int = 0, state=None):
    """Causal FLARE over N tokens: y_t uses keys/values of tokens <= t only.
    Returns (y [B,H,N,D], state) where state = (mu, den, num) continues the recurrence.
    `chunk` is the length of the token segments the matrix-core path runs in parallel
    (0 = chosen from B*H and N); the result depends on it only through rounding."""
    return _causal_call("prefill", q, k, v, scale, chunk, state)


def flare_causal_decode(q, k, v, state, scale: float = 1.0, inplace: bool = False, workspace=None, out=None):
    """n recurrent single-token steps in one launch; k, v are [B,H,n,D].

    By default the incoming state is left as it was and a new one is returned.  inplace=True advances the given
    state tensors themselves (contiguous fp32 on the device; returned again), `workspace` (from causal_workspace)
    and `out` ([B,H,n,D]) let a decode loop reuse its buffers, so that a step allocates nothing and can be
    captured in a HIP graph.  In-place calls need a shape the kernels take directly (M in {128, 256} with
    D in {32, 64} for 16-bit inputs, or anything the fp32 kernel takes)."""
    return _causal_call("decode", q, k, v, scale, 0, state, inplace=inplace, workspace=workspace, out=out)


def flare_causal_decode_step(q, k_t, v_t, state, scale: float = 1.0, inplace: bool = False, workspace=None, out=None):
    """One token: k_t, v_t are [B,H,D] or [B,H,1,D] (out, if given, [B,H,1,D]).  See flare_causal_decode."""
    squeeze = k_t.dim() == 3
    if squeeze:
        k_t, v_t = k_t.unsqueeze(2), v_t.unsqueeze(2)
    y, st = _causal_call("decode", q, k_t, v_t, scale, 0, state, inplace=inplace, workspace=workspace, out=out)
    return (y.squeeze(2) if squeeze else y), st


# --------------------------------------------------------------------------------------
# causal linear attention
# --------------------------------------------------------------------------------------
def _causal_linear_desc(q, k, v, y, n_segs=0, force_generic=False):
    B, H, N, Dk = q.shape
    d = _lib.FlareCausalLinearDesc()
    d.B, d.H, d.N, d.Dk, d.Dv = B, H, N, Dk, v.shape[-1]
    d.dtype = _dtype_code(q)
    d.n_segs = int(n_segs)
    d.flags = _lib.FLAG_FORCE_GENERIC if force_generic else 0
    d.q_stride, d.k_stride, d.v_stride, d.y_stride = _s3(q), _s3(k), _s3(v), _s3(y)
    return d


def _causal_linear_forward(q, k, v, n_segs: int = 0, force_generic: bool = False):
    """(y, the launch's workspace: the segments' states, which the backward starts from)."""
    _require_cuda(q, k, v)
    lib = _lib.load()
    if q.dim() != 4 or q.shape != k.shape:
        raise ValueError(f"Q, K must have the same shape [B,H,N,Dk]. Got Q.shape={tuple(q.shape)}, K.shape={tuple(k.shape)}")
    B, H, N, Dk = q.shape
    if v.dim() != 4 or v.shape[:3] != (B, H, N):
        raise ValueError(f"V must have shape ({B}, {H}, {N}, Dv). Got V.shape={tuple(v.shape)}")
    if not (q.dtype == k.dtype == v.dtype):
        raise ValueError("Q, K, V must share one dtype")
    q, k, v = _rows_last_contig(q), _rows_last_contig(k), _rows_last_contig(v)
    y = torch.empty((B, H, N, v.shape[-1]), dtype=q.dtype, device=q.device)
    d = _causal_linear_desc(q, k, v, y, n_segs, force_generic)
    with _on_device(q.device):
        need = C.c_size_t(0)
        _lib.check(lib.flare_causal_linear_workspace_bytes(C.byref(d), C.byref(need)),
                   "flare_causal_linear_workspace_bytes")
        ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=q.device)
        rc = lib.flare_causal_linear_fwd(C.byref(d), _ptr(q), _ptr(k), _ptr(v), _ptr(y), _ptr(ws), ws.numel(),
                                         C.c_void_p(_stream_ptr(q.device)))
    _lib.check(rc, "flare_causal_linear_fwd")
    return y, ws


class _CausalLinearFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v):
        q, k, v = _rows_last_contig(q), _rows_last_contig(k), _rows_last_contig(v)
        y, ws = _causal_linear_forward(q, k, v)
        # rows off the 16-byte grid took the FMA kernels, which leave other states behind: the backward, which may get these tensors
        # back on another grid (a saved-tensor hook), must not start from them
        ctx.states = not any(t.data_ptr() % 16 or any(s % 8 for s in t.stride()[:3]) for t in (q, k, v))
        ctx.save_for_backward(q, k, v, ws)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, gy):
        # Every gradient is a causal linear attention again (the same kernels, the last two over the reversed token axis):
        #   dq_t   = (1/N) sum_{tau <= t} <gy_t, v_tau> k_tau
        #   dk_tau = (1/N) sum_{t >= tau} <v_tau, gy_t> q_t
        #   dv_tau = (1/N) sum_{t >= tau} <k_tau, q_t> gy_t
        q, k, v, fwd_ws = ctx.saved_tensors
        q, k, v = _rows_last_contig(q), _rows_last_contig(k), _rows_last_contig(v)
        gy = gy.to(q.dtype)
        if gy.stride(-1) != 1 or any(s % 8 for s in gy.stride()[:3]) or gy.data_ptr() % 16 or gy.stride(2) < gy.shape[-1]:
            gy = gy.contiguous()
        grads = [torch.empty(t.shape, dtype=q.dtype, device=q.device) if need else None
                 for t, need in zip((q, k, v), ctx.needs_input_grad)]
        ws = torch.empty_like(fwd_ws)
        d = _causal_linear_desc(q, k, v, v)
        with _on_device(q.device):
            rc = _lib.load().flare_causal_linear_bwd(C.byref(d), _ptr(q), _ptr(k), _ptr(v), _ptr(gy), _s3(gy),
                                                     _ptr(fwd_ws) if ctx.states else None, *(_ptr(t) for t in grads), _ptr(ws), ws.numel(),
                                                     C.c_void_p(_stream_ptr(q.device)))
        _lib.check(rc, "flare_causal_linear_bwd")
        return tuple(grads)


def causal_linear_attention(q, k, v, n_segs: int = 0, force_generic: bool = False):
    """y_t = (1/N) sum_{tau<=t} <q_t,k_tau> v_tau for q,k [B,H,N,Dk], v [B,H,N,Dv] -> [B,H,N,Dv]
    (lra/models/triton/causal_linear.py:317-336).  n_segs = token segments run in parallel (0 = auto).
    Dk in {64, 128} with 16-byte aligned rows runs on the matrix cores: bf16 / f16 with Dv in {32, 64, 128} (products
    in the input type, fp32 accumulation and state), fp32 with Dv in {32, 64} (fp32 products); everything else, and
    force_generic=True, as fp32 FMA loops."""
    if n_segs == 0 and not force_generic and torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v)):
        return _CausalLinearFn.apply(q, k, v)
    return _causal_linear_forward(q, k, v, n_segs, force_generic)[0]


class CausalLinear:
    """Call-compatible stand-in for lra/models/triton/causal_linear.py:23 `CausalLinear`:
    `CausalLinear.apply(Q, K, V) -> Y`.  The HIP kernels need no N % 64 == 0."""

    @staticmethod
    def apply(Q, K, V):
        return causal_linear_attention(Q, K, V)


# --------------------------------------------------------------------------------------
# triple attention
# --------------------------------------------------------------------------------------
def _triple_desc(q1, q2, k1, k2, v, out, feature_map=False, normalize=False, n_splits=0):
    d = FlareTripleDesc()
    d.B, d.H, d.N, d.Dq = q1.shape
    d.Dv = v.shape[-1]
    d.dtype = _dtype_code(q1)
    d.feature_map, d.normalize, d.n_splits = int(feature_map), int(normalize), int(n_splits)
    d.q1_stride, d.q2_stride, d.k1_stride, d.k2_stride = _s3(q1), _s3(q2), _s3(k1), _s3(k2)
    d.v_stride, d.o_stride = _s3(v), _s3(out)
    return d


def _triple_forward(q1, q2, k1, k2, v, feature_map: bool, normalize: bool, n_splits: int = 0):
    _require_cuda(q1, q2, k1, k2, v)
    lib = _lib.load()
    if not (q1.shape == q2.shape == k1.shape == k2.shape):
        raise ValueError("q1, q2, k1, k2 must share one shape [B,H,N,Dq]")
    if v.shape[:-1] != q1.shape[:-1] or q1.dim() != 4:
        raise ValueError("v must be [B,H,N,Dv] with the same B,H,N as q1")
    if not (q1.dtype == q2.dtype == k1.dtype == k2.dtype == v.dtype):
        raise TypeError("all five inputs must share a dtype")
    q1, q2, k1, k2, v = (_rows_last_contig(t) for t in (q1, q2, k1, k2, v))
    B, H, N, Dq = q1.shape
    Dv = v.shape[-1]
    Dqp, Dvp = -(-Dq // 16) * 16, -(-Dv // 16) * 16
    if (Dqp, Dvp) != (Dq, Dv) and q1.dtype in (torch.bfloat16, torch.float16) and max(Dqp, Dvp) <= 64:
        # The matrix-core kernels take head dims that are multiples of 16 (up to 64).  Any other head dim up to 64:
        # features first (elu + 1, rounded to the element type as the kernels do when they stage a tile), then zero
        # columns up to the next multiple of 16 (they add nothing to either contraction, nor to the normaliser).
        if feature_map:
            q1, q2, k1, k2 = ((torch.nn.functional.elu(t.float()) + 1.0).to(t.dtype) for t in (q1, q2, k1, k2))
        if Dqp != Dq:
            q1, q2, k1, k2 = (_pad_last(t, Dqp - Dq) for t in (q1, q2, k1, k2))
        vp = _pad_last(v, Dvp - Dv) if Dvp != Dv else v
        state, out = _triple_forward(q1, q2, k1, k2, vp, False, normalize, n_splits)
        return state[:, :, :Dq, :Dv, :Dq].contiguous(), out[..., :Dv].contiguous()
    state = torch.empty((B, H, Dq, Dv, Dq), dtype=torch.float32, device=q1.device)
    out = torch.empty((B, H, N, Dv), dtype=q1.dtype, device=q1.device)
    d = _triple_desc(q1, q2, k1, k2, v, out, feature_map, normalize, n_splits)
    need = C.c_size_t(0)
    _lib.check(lib.flare_triple_workspace_bytes(C.byref(d), C.byref(need)), "flare_triple_workspace_bytes")
    ws = torch.empty(max(int(need.value), 16), dtype=torch.uint8, device=q1.device)
    with _on_device(q1.device):
        rc = lib.flare_triple_fwd(C.byref(d), _ptr(q1), _ptr(q2), _ptr(k1), _ptr(k2), _ptr(v), _ptr(state),
                                  _ptr(out), _ptr(ws), ws.numel(), C.c_void_p(_stream_ptr(q1.device)))
    _lib.check(rc, "flare_triple_fwd")
    return state, out


class _TripleFn(torch.autograd.Function):
    """(STATE, O) = triple attention with the gradients of lra/models/triton/triple.py:124-135.  Every
    gradient is again a state or an output contraction, so for Dq == Dv the backward runs on the
    HIP kernels of the forward with permuted states (flare_triple_bwd); otherwise it is the reference's einsum formulas."""

    @staticmethod
    def forward(ctx, q1, q2, k1, k2, v):
        ctx.set_materialize_grads(False)
        q1, q2, k1, k2, v = (_rows_last_contig(t) for t in (q1, q2, k1, k2, v))
        state, out = _triple_forward(q1, q2, k1, k2, v, False, False)
        ctx.save_for_backward(q1, q2, k1, k2, v, state)
        return state, out

    @staticmethod
    @once_differentiable
    def backward(ctx, dstate, dout):
        *rows, state = ctx.saved_tensors
        q1, q2, k1, k2, v = (_rows_last_contig(t) for t in rows)      # a saved-tensor hook may change the memory order
        state = state.contiguous()
        N = q1.shape[2]
        dt = q1.dtype
        if dout is None:
            dout = torch.zeros_like(v)
        if q1.shape[-1] == v.shape[-1]:
            lib = _lib.load()
            do = _rows_last_contig(dout.to(dt))
            grads = [torch.empty(t.shape, dtype=dt, device=t.device) for t in (q1, q2, k1, k2, v)]
            if dstate is not None:
                dstate = dstate.to(torch.float32).contiguous()
            d = _triple_desc(q1, q2, k1, k2, v, do)
            need = C.c_size_t(0)
            _lib.check(lib.flare_triple_bwd_workspace_bytes(C.byref(d), C.byref(need)), "flare_triple_bwd_workspace_bytes")
            ws = torch.empty(int(need.value), dtype=torch.uint8, device=q1.device)
            with _on_device(q1.device):
                rc = lib.flare_triple_bwd(C.byref(d), _ptr(q1), _ptr(q2), _ptr(k1), _ptr(k2), _ptr(v), _ptr(state), _ptr(dstate),
                                          _ptr(do), *(_ptr(g) for g in grads), _ptr(ws), ws.numel(), C.c_void_p(_stream_ptr(q1.device)))
            _lib.check(rc, "flare_triple_bwd")
            return tuple(grads)
        f = lambda t: t.float()
        do = f(dout)
        dq1 = torch.einsum("bhnj,bhijk,bhnk->bhni", do, state, f(q2))
        dq2 = torch.einsum("bhnj,bhni,bhijk->bhnk", do, f(q1), state)
        ds = torch.einsum("bhnj,bhni,bhnk->bhijk", do, f(q1), f(q2))
        if dstate is not None:
            ds = ds + dstate.float()
        dk1 = torch.einsum("bhijk,bhnj,bhnk->bhni", ds, f(v), f(k2)) / N
        dk2 = torch.einsum("bhijk,bhni,bhnj->bhnk", ds, f(k1), f(v)) / N
        dv = torch.einsum("bhijk,bhni,bhnk->bhnj", ds, f(k1), f(k2)) / N
        return dq1.to(dt), dq2.to(dt), dk1.to(dt), dk2.to(dt), dv.to(dt)


def triple_attention(q1, q2, k1, k2, v, normalize: bool = False, feature_map: Optional[str] = None,
                     n_splits: int = 0):
    """Third-order linear attention (lra/models/backends.py:1285-1292 of the reference).

    Returns (state [B,H,Dq,Dv,Dq] fp32, out [B,H,N,Dv]).  feature_map=None expects inputs that
    already went through the kernel map (as TripleAttention.forward does at backends.py:1258);
    feature_map='elu' applies elu(x)+1 to q1,q2,k1,k2 inside the kernels.
    normalize=True divides out by the matching normaliser (same contraction with v == 1).
    Differentiable in all five inputs in every mode.
    """
    if feature_map not in (None, "identity", "elu"):
        raise ValueError("feature_map must be None, 'identity' or 'elu'")
    needs_grad = torch.is_grad_enabled() and any(t.requires_grad for t in (q1, q2, k1, k2, v))
    if needs_grad:
        # Under autograd the feature map is applied with torch ops in front of the kernels (where the reference applies it,
        # backends.py:1258) and the normaliser is formed with two small einsums behind them, so that both differentiate
        # through torch while the two contractions and their gradients stay on the HIP kernels.
        if feature_map == "elu":
            q1, q2, k1, k2 = (torch.nn.functional.elu(t) + 1 for t in (q1, q2, k1, k2))
        state, out = _TripleFn.apply(q1, q2, k1, k2, v)
        if normalize:
            kk = torch.einsum("bhni,bhnk->bhik", k1.float(), k2.float()) / k1.shape[-2]
            den = torch.einsum("bhni,bhik,bhnk->bhn", q1.float(), kk, q2.float())
            out = (out.float() / den.unsqueeze(-1)).to(out.dtype)
        return state, out
    return _triple_forward(q1, q2, k1, k2, v, feature_map == "elu", normalize, n_splits)


class TripleAttentionFunction:
    """Call-compatible stand-in for lra/models/triton/triple.py:27 `TripleAttentionFunction`:
    `TripleAttentionFunction.apply(Q1, Q2, K1, K2, V) -> (STATE, O)`, differentiable like the original."""

    @staticmethod
    def apply(Q1, Q2, K1, K2, V):
        return triple_attention(Q1, Q2, K1, K2, V)
