"""Host-side checks of the C-ABI that need no GPU: the library loads, exports every symbol
include/flare_hip.h declares, and rejects bad requests before anything is launched."""
import ctypes as C
import os
import re

import pytest
import torch

import flare_py_amd as F
from flare_py_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _mixer_desc(B=1, H=2, N=128, M=64, D=32, dtype=_lib.DT_BF16, scale=1.0):
    d = _lib.FlareMixerDesc()
    d.B, d.H, d.N, d.M, d.D, d.dtype, d.scale = B, H, N, M, D, dtype, scale
    d.q_stride = _lib.I3(0, M * D, D)
    d.k_stride = d.v_stride = d.y_stride = _lib.I3(H * N * D, N * D, D)
    return d


def test_header_symbols_all_exported():
    text = open(os.path.join(ROOT, "include", "flare_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    declared = set(re.findall(r"\b(flare_[a-z_]+)\s*\(", text))
    assert declared, "no declarations parsed"
    lib = _lib.load()
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in flare_hip.h but not exported"
    assert declared == set(_lib.SYMBOLS), "ctypes binding and header disagree"
    assert lib.flare_abi_version() == _lib.ABI_VERSION == 2


def test_struct_sizes_match_header_layout():
    assert C.sizeof(_lib.FlareMixerDesc) == 10 * 4 + 4 * 24 + 16       # + dropout_p, reserved2, dropout_seed
    assert C.sizeof(_lib.FlareCausalDesc) == 10 * 4 + 4 * 24
    assert C.sizeof(_lib.FlareTripleDesc) == 10 * 4 + 6 * 24


def test_workspace_query_and_kernel_choice():
    lib = _lib.load()
    n = C.c_size_t(0)
    d = _mixer_desc()
    assert lib.flare_mixer_workspace_bytes(C.byref(d), C.byref(n)) == 0 and n.value > 0
    assert lib.flare_mixer_kernel_name(C.byref(d)) == b"mfma_bf16"
    d.flags = _lib.FLAG_FORCE_GENERIC
    assert lib.flare_mixer_kernel_name(C.byref(d)) == b"generic"
    assert lib.flare_mixer_kernel_name(C.byref(_mixer_desc(dtype=_lib.DT_F32))) == b"generic"
    assert lib.flare_mixer_kernel_name(C.byref(_mixer_desc(M=16, D=8))) == b"generic"
    assert lib.flare_mixer_kernel_name(C.byref(_mixer_desc(dtype=_lib.DT_F16))) == b"mfma_f16"


@pytest.mark.parametrize("field,value,code", [
    ("N", 0, _lib.FLARE_EINVAL), ("M", -1, _lib.FLARE_EINVAL), ("D", 256, _lib.FLARE_EUNSUPPORTED),
    ("dtype", 7, _lib.FLARE_EINVAL), ("scale", 0.0, _lib.FLARE_EINVAL), ("n_splits", -2, _lib.FLARE_EINVAL),
])
def test_bad_descriptor_rejected(field, value, code):
    lib = _lib.load()
    d = _mixer_desc()
    setattr(d, field, value)
    n = C.c_size_t(0)
    assert lib.flare_mixer_workspace_bytes(C.byref(d), C.byref(n)) == code
    assert _lib.last_error() != ""


def test_null_pointers_and_workspace_rejected_before_launch():
    lib = _lib.load()
    d = _mixer_desc()
    one = C.c_void_p(16)  # never dereferenced: validation fails first
    assert lib.flare_mixer_fwd(C.byref(d), None, one, one, None, one, None, one, 1 << 30, None) == _lib.FLARE_EINVAL
    assert lib.flare_mixer_fwd(C.byref(d), one, one, one, None, one, None, None, 0, None) == _lib.FLARE_EWORKSPACE
    assert lib.flare_mixer_fwd(C.byref(d), one, one, one, None, one, None, one, 8, None) == _lib.FLARE_EWORKSPACE
    assert "needed" in _lib.last_error()
    assert lib.flare_gather_fwd(C.byref(d), one, one, one, None, None, None, one, 1 << 30, None) == _lib.FLARE_EINVAL
    assert lib.flare_scatter_fwd(C.byref(d), one, one, None, None, one, None) == _lib.FLARE_EINVAL
    d.k_stride = _lib.I3(0, 0, 3)  # row stride < D
    assert lib.flare_scatter_fwd(C.byref(d), one, one, one, None, one, None) == _lib.FLARE_EINVAL
    assert lib.flare_mixer_workspace_bytes(None, C.byref(C.c_size_t(0))) == _lib.FLARE_EINVAL


def test_causal_and_triple_validation():
    lib = _lib.load()
    one = C.c_void_p(16)
    c = _lib.FlareCausalDesc()
    c.B, c.H, c.N, c.M, c.D, c.dtype, c.scale = 1, 1, 8, 16, 16, 0, 1.0
    c.q_stride = _lib.I3(0, 256, 16)
    c.k_stride = c.v_stride = c.y_stride = _lib.I3(128, 128, 16)
    assert lib.flare_causal_prefill_fwd(C.byref(c), one, one, one, one, None, one, one, None, 0, None) == _lib.FLARE_EINVAL
    c.M, c.D = 4096, 128
    n = C.c_size_t(0)
    assert lib.flare_causal_workspace_bytes(C.byref(c), C.byref(n)) == _lib.FLARE_EUNSUPPORTED
    t = _lib.FlareTripleDesc()
    t.B, t.H, t.N, t.Dq, t.Dv, t.dtype = 1, 1, 64, 16, 16, 1
    assert lib.flare_triple_workspace_bytes(C.byref(t), C.byref(n)) == 0 and n.value > 0
    assert lib.flare_triple_fwd(C.byref(t), one, one, one, one, one, one, one, one, 4, None) == _lib.FLARE_EWORKSPACE
    t.Dq = 128
    assert lib.flare_triple_workspace_bytes(C.byref(t), C.byref(n)) == _lib.FLARE_EUNSUPPORTED
    t.Dq, t.feature_map = 16, 5
    assert lib.flare_triple_workspace_bytes(C.byref(t), C.byref(n)) == _lib.FLARE_EINVAL


def test_python_api_fails_loudly_on_cpu_tensors():
    q = torch.randn(2, 4, 8)
    k = torch.randn(1, 2, 16, 8)
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        F.flare_multihead_mixer(q, k, k)
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        F.triple_attention(k, k, k, k, k)
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        F.flare_causal_prefill(q, k, k)


def test_status_to_exception_mapping():
    _lib.load().flare_mixer_workspace_bytes(None, None)
    with pytest.raises(ValueError):
        _lib.check(_lib.FLARE_EINVAL, "x")
    with pytest.raises(NotImplementedError):
        _lib.check(_lib.FLARE_EUNSUPPORTED, "x")
    with pytest.raises(RuntimeError):
        _lib.check(_lib.FLARE_EHIP, "x")


def test_new_struct_sizes_and_entry_point_validation():
    assert C.sizeof(_lib.FlareCausalLinearDesc) == 8 * 4 + 4 * 24
    assert C.sizeof(_lib.FlareMlpDesc) == 8 + 12 * 4 + 3 * 8
    lib = _lib.load()
    # fused MLP: argument checks happen before anything is launched
    m = _lib.FlareMlpDesc()
    m.T, m.C, m.L, m.w_dtype = 16, 128, 2, _lib.DT_BF16
    m.x_stride = m.y_stride = 128
    assert lib.flare_mlp_fwd(m, None, None, None, None, None, None, None, None) == _lib.FLARE_EINVAL
    assert "must not be NULL" in _lib.last_error()
    m.C = 48
    assert lib.flare_mlp_fwd(m, None, None, None, None, None, None, None, None) == _lib.FLARE_EUNSUPPORTED
    m.C, m.L = 128, 0
    assert lib.flare_mlp_fwd(m, None, None, None, None, None, None, None, None) == _lib.FLARE_EINVAL
    m.L, m.w_dtype = 2, _lib.DT_F32
    assert lib.flare_mlp_fwd(m, None, None, None, None, None, None, None, None) == _lib.FLARE_EINVAL
    # narrow first / last layers: widths above 4, a norm in front of a lifting layer, expand mode and a
    # residual next to a narrow output are refused (fake non-NULL pointers: nothing is dereferenced before the checks)
    m.w_dtype = _lib.DT_BF16
    fake = C.c_void_p(4096)
    io = lambda i, o, res=None: lib.flare_mlp_io_fwd(m, i, 1, fake, fake, o, fake, fake, None, fake, None, res, fake, None)
    assert io(5, 0) == _lib.FLARE_EINVAL and "in_dim and out_dim" in _lib.last_error()
    assert io(0, 7) == _lib.FLARE_EINVAL
    m.norm = 1
    assert io(3, 0) == _lib.FLARE_EINVAL and "norm" in _lib.last_error()
    m.norm, m.flags = 0, _lib.MLP_EXPAND
    assert io(3, 0) == _lib.FLARE_EINVAL and "EXPAND" in _lib.last_error()
    m.flags = 0
    assert io(0, 2, fake) == _lib.FLARE_EINVAL and "res must be NULL" in _lib.last_error()
    m.x_stride = 2
    assert io(3, 0) == _lib.FLARE_EINVAL and "x_stride" in _lib.last_error()
    # head-padded rows: head dims 4 and 8 only, not next to in_dim / out_dim, and rows wide enough for the padding
    m.x_stride = 128
    m.flags = (12 // 4) << 8
    assert lib.flare_mlp_fwd(m, fake, fake, None, fake, None, None, fake, None) == _lib.FLARE_EINVAL and "head dim" in _lib.last_error()
    m.flags = (8 // 4) << 12
    assert io(3, 0) == _lib.FLARE_EINVAL and "head dim" in _lib.last_error()
    assert lib.flare_mlp_fwd(m, fake, fake, None, fake, None, None, fake, None) == _lib.FLARE_EINVAL and "row width" in _lib.last_error()
    m.flags = 0
    # causal linear attention
    c = _lib.FlareCausalLinearDesc()
    c.B, c.H, c.N, c.Dk, c.Dv, c.dtype = 1, 2, 100, 32, 16, _lib.DT_F32
    c.q_stride = c.k_stride = _lib.I3(6400, 3200, 32)
    c.v_stride = c.y_stride = _lib.I3(3200, 1600, 16)
    need = C.c_size_t(0)
    assert lib.flare_causal_linear_workspace_bytes(c, C.byref(need)) == _lib.FLARE_OK and need.value > 0
    assert lib.flare_causal_linear_fwd(c, None, None, None, None, None, 0, None) == _lib.FLARE_EINVAL
    c.Dk = 200
    assert lib.flare_causal_linear_workspace_bytes(c, C.byref(need)) == _lib.FLARE_EUNSUPPORTED
    # mixer backward: supported shapes only, workspace checked
    d = _mixer_desc(M=128, D=32)
    assert lib.flare_mixer_bwd_workspace_bytes(d, C.byref(need)) == _lib.FLARE_OK and need.value > 0
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(dtype=_lib.DT_F32), C.byref(need)) == _lib.FLARE_OK     # fp32 kernels
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(dtype=_lib.DT_F32, M=40), C.byref(need)) == _lib.FLARE_EUNSUPPORTED
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(dtype=_lib.DT_F32, D=24), C.byref(need)) == _lib.FLARE_EUNSUPPORTED
    # the halves' backward: every dtype (16-bit without dropout), arguments checked before anything is launched
    f = _mixer_desc(dtype=_lib.DT_F32)
    assert lib.flare_gather_bwd(d, *([None] * 9), None, 0, None) == _lib.FLARE_EWORKSPACE
    d.dropout_p = 0.25
    assert lib.flare_gather_bwd(d, *([None] * 9), None, 0, None) == _lib.FLARE_EUNSUPPORTED and "dropout" in _lib.last_error()
    d.dropout_p = 0.0
    assert lib.flare_gather_bwd(f, *([None] * 9), None, 0, None) == _lib.FLARE_EWORKSPACE
    assert lib.flare_scatter_bwd(f, *([None] * 6), None, None, None, None, None, 0, None) == _lib.FLARE_EWORKSPACE
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(M=256, D=64), C.byref(need)) == _lib.FLARE_OK      # one LDS-full exactly
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(M=1024, D=64), C.byref(need)) == _lib.FLARE_OK     # four chunks of latents
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(M=2048, D=64), C.byref(need)) == _lib.FLARE_EUNSUPPORTED
    assert lib.flare_mixer_bwd_workspace_bytes(_mixer_desc(M=48, D=32), C.byref(need)) == _lib.FLARE_EUNSUPPORTED
    assert lib.flare_mixer_bwd(d, *([None] * 8), None, None, None, None, None, 0, None) == _lib.FLARE_EINVAL
    assert lib.flare_scatter_fwd_lse(d, None, None, None, None, None, None, None) == _lib.FLARE_EINVAL


@pytest.mark.parametrize("Cdim,L", [(32, 1), (64, 3), (128, 8)])
def test_both_weight_images_from_one_gather_equal_the_two_single_ones(Cdim, L):
    """A training step builds the image of the weights and of their transposes in one indexed read; each has to be what
    mlp_weight_image (checked against the header's formula below) gives for the matrix and for its transpose."""
    from flare_py_amd import fused
    w = torch.randn(L, Cdim, Cdim, generator=torch.Generator().manual_seed(Cdim + L)).to(torch.bfloat16)
    img, img_t = fused.mlp_weight_images(w)
    assert img.is_contiguous() and img_t.is_contiguous() and img.shape == img_t.shape == (L, Cdim * Cdim)
    assert torch.equal(img, fused.mlp_weight_image(w))
    assert torch.equal(img_t, fused.mlp_weight_image(w.transpose(1, 2).contiguous()))


@pytest.mark.parametrize("Cdim", [32, 64, 128])
def test_mlp_weight_image_follows_the_header_formula(Cdim):
    """fused.mlp_weight_image against include/flare_hip.h's position formula, element by element in plain loops:
    the image is a permutation inside each row, and a 16-byte piece holds four columns of one 8-column block and the
    same four of the block two further on."""
    from flare_py_amd import fused
    shift = {128: 0, 64: 1, 32: 2}[Cdim]
    w = torch.arange(2 * Cdim * Cdim, dtype=torch.float32).view(2, Cdim, Cdim)
    img = fused.mlp_weight_image(w).view(2, Cdim * Cdim)
    seen = set()
    for row in range(Cdim):
        for col in range(Cdim):
            ch, j = col // 8, col % 8
            key = (row % 16) >> shift
            pos = row * Cdim + 8 * ((4 * (ch // 4) + 2 * (ch % 2) + j // 4) ^ key) + 4 * ((ch % 4) // 2) + j % 4
            assert pos // Cdim == row and pos not in seen
            seen.add(pos)
            for l in range(2):
                assert img[l, pos] == w[l, row, col]
    assert len(seen) == Cdim * Cdim
    piece = img[0].view(Cdim, Cdim // 8, 8)[5].long() - 5 * Cdim          # columns held by row 5's pieces
    for p in piece:
        lo, hi = p[:4].tolist(), p[4:].tolist()
        assert lo == list(range(lo[0], lo[0] + 4)) and lo[0] % 4 == 0
        assert hi == [c + 16 for c in lo]


def test_mlp_bwd_validation():
    lib = _lib.load()
    m = _lib.FlareMlpDesc()
    m.T, m.C, m.L = 64, 128, 2
    m.x_dtype = m.y_dtype = m.w_dtype = _lib.DT_BF16
    m.norm, m.act, m.eps = 1, 0, 1e-5      # layer norm, tanh gelu
    m.x_stride = m.y_stride = 128
    fake = C.c_void_p(4096)
    odd = C.c_void_p(4100)
    ff = fake
    rows = C.c_int32(0)
    assert lib.flare_mlp_bwd_partial_rows(m, C.byref(rows)) == _lib.FLARE_OK and rows.value == 1
    m.T = 1 << 20
    assert lib.flare_mlp_bwd_partial_rows(m, C.byref(rows)) == _lib.FLARE_OK and 1 <= rows.value <= 4096
    big = rows.value
    m.T = 1 << 22
    assert lib.flare_mlp_bwd_partial_rows(m, C.byref(rows)) == _lib.FLARE_OK and rows.value == big     # capped by the CU count
    assert lib.flare_mlp_bwd_partial_rows(m, None) == _lib.FLARE_EINVAL
    m.T = 64

    def call(x=fake, dy=fake, gamma=ff, dn=fake, stats=ff, gb=ff):
        return lib.flare_mlp_bwd(m, x, dy, fake, fake, ff, gamma, ff, 0, fake, fake, fake, dn, stats, gb, None, None)

    assert lib.flare_mlp_bwd(None, *([None] * 7), 0, *([None] * 8)) == _lib.FLARE_EINVAL
    # add_dy is a set of two bits (add dy, accumulate into dx); anything else is refused before a launch
    assert lib.flare_mlp_bwd(m, fake, fake, fake, fake, ff, ff, ff, 4, fake, fake, fake, fake, ff, ff, None, None) == _lib.FLARE_EINVAL
    assert "unknown bits" in _lib.last_error()
    assert call(x=None) == _lib.FLARE_EINVAL and "must not be NULL" in _lib.last_error()
    assert call(gamma=None) == _lib.FLARE_EINVAL and "norm" in _lib.last_error()
    assert call(gb=None) == _lib.FLARE_EINVAL and "norm" in _lib.last_error()
    assert call(x=odd) == _lib.FLARE_EINVAL and "16-byte" in _lib.last_error()
    assert call(dn=odd) == _lib.FLARE_EINVAL and "16-byte" in _lib.last_error()
    m.L = 6
    assert call() == _lib.FLARE_EUNSUPPORTED and "at most 5 layers" in _lib.last_error()
    m.C = 64
    m.x_stride = 62
    assert call() == _lib.FLARE_EINVAL and "row stride" in _lib.last_error()
    m.x_stride = 64
    m.y_stride = 66
    assert call() == _lib.FLARE_EINVAL and "y_stride" in _lib.last_error()
    m.y_stride = 64
    m.L = 9
    assert call() == _lib.FLARE_EUNSUPPORTED and "at most 8 layers" in _lib.last_error()
    m.L = 2
    m.C = 48
    assert call() == _lib.FLARE_EUNSUPPORTED and "32, 64 and 128" in _lib.last_error()
    m.C = 128
    m.x_stride = m.y_stride = 128
    m.flags = _lib.MLP_EXPAND
    assert call() == _lib.FLARE_EUNSUPPORTED and "flags must be 0" in _lib.last_error()
    m.flags = 0
    m.w_dtype = _lib.DT_F32
    assert call() == _lib.FLARE_EINVAL and "w_dtype" in _lib.last_error()
    m.w_dtype = _lib.DT_BF16
    m.act = 7
    assert call() == _lib.FLARE_EINVAL and "activation" in _lib.last_error()
    m.act, m.eps = 0, -1.0
    assert call() == _lib.FLARE_EINVAL and "eps" in _lib.last_error()


def test_mlp_wgrad_validation():
    lib = _lib.load()
    m = _lib.FlareMlpDesc()
    m.T, m.C, m.L = 262144, 128, 5
    m.w_dtype = _lib.DT_BF16
    fake, odd = C.c_void_p(4096), C.c_void_p(4100)
    parts = C.c_int32(0)
    assert lib.flare_mlp_wgrad_partials(m, C.byref(parts)) == _lib.FLARE_OK and 1 <= parts.value <= 1024
    big = parts.value
    m.T = 100
    assert lib.flare_mlp_wgrad_partials(m, C.byref(parts)) == _lib.FLARE_OK and parts.value == 1
    m.C = 32            # eight waves split a token tile: eight partials per token range
    assert lib.flare_mlp_wgrad_partials(m, C.byref(parts)) == _lib.FLARE_OK and parts.value == 8
    m.C, m.T = 128, 262144
    assert lib.flare_mlp_wgrad_partials(m, None) == _lib.FLARE_EINVAL
    assert lib.flare_mlp_wgrad(m, None, 0, fake, 0, fake, None, None, None, None) == _lib.FLARE_EINVAL and "must not be NULL" in _lib.last_error()
    assert lib.flare_mlp_wgrad(m, fake, 0, fake, 0, odd, None, None, None, None) == _lib.FLARE_EINVAL and "16-byte" in _lib.last_error()
    assert lib.flare_mlp_wgrad(m, fake, 0, fake, 0, fake, None, fake, fake, None) == _lib.FLARE_EINVAL and "db needs db_part" in _lib.last_error()
    m.C = 96
    assert lib.flare_mlp_wgrad(m, fake, 0, fake, 0, fake, None, None, None, None) == _lib.FLARE_EUNSUPPORTED
    m.C, m.w_dtype = 128, _lib.DT_F32
    assert lib.flare_mlp_wgrad(m, fake, 0, fake, 0, fake, None, None, None, None) == _lib.FLARE_EINVAL and "w_dtype" in _lib.last_error()
    m.w_dtype = _lib.DT_BF16
    assert lib.flare_mlp_wgrad(m, fake, 4, fake, 0, fake, None, None, None, None) == _lib.FLARE_EINVAL and "layer strides" in _lib.last_error()
    m.L = 0
    assert lib.flare_mlp_wgrad_partials(m, C.byref(parts)) == _lib.FLARE_EINVAL
    assert big >= 64


def test_mlp_expand_bwd_validation():
    lib = _lib.load()
    m = _lib.FlareMlpDesc()
    m.T, m.C, m.L, m.flags = 64, 128, 8, _lib.MLP_EXPAND
    m.x_dtype = m.y_dtype = m.w_dtype = _lib.DT_BF16
    m.norm, m.act, m.eps = 1, 0, 1e-5
    m.x_stride = m.y_stride = 128
    fake, odd = C.c_void_p(4096), C.c_void_p(4100)

    def call(x=fake, h=fake, gamma=fake, dn=fake):
        return lib.flare_mlp_expand_bwd(m, x, fake, fake, fake, fake, gamma, fake, 0, fake, fake, fake, h, fake, dn, fake, fake, None, None)

    assert call(x=None) == _lib.FLARE_EINVAL and "must not be NULL" in _lib.last_error()
    assert call(h=odd) == _lib.FLARE_EINVAL and "16-byte" in _lib.last_error()
    assert call(gamma=None) == _lib.FLARE_EINVAL and "norm" in _lib.last_error()
    m.L = 7
    assert call() == _lib.FLARE_EUNSUPPORTED and "2 E tiles" in _lib.last_error()
    m.L = 18
    assert call() == _lib.FLARE_EUNSUPPORTED
    m.L, m.flags = 8, 0
    assert call() == _lib.FLARE_EINVAL and "FLARE_MLP_EXPAND" in _lib.last_error()
    m.flags, m.C = _lib.MLP_EXPAND, 96
    assert call() == _lib.FLARE_EUNSUPPORTED


def test_few_token_limits_agree_with_the_library():
    from flare_py_amd import fused

    lib = _lib.load()
    for Cdim in (32, 64, 128):
        for L in (1, 5, 6, 8, 9):
            for T in (1, 16, 17, 12288, 12289, 16384, 16385, 1 << 20):
                m = _lib.FlareMlpDesc()
                m.T, m.C, m.L, m.w_dtype = T, Cdim, L, _lib.DT_BF16
                assert lib.flare_mlp_few(C.byref(m)) == fused._few(T, Cdim, L), (Cdim, L, T)
    m.flags = _lib.MLP_EXPAND
    m.T = 16
    assert lib.flare_mlp_few(C.byref(m)) == 0


def test_few_token_question_at_unsupported_widths():
    """No, and no error either: the launch itself refuses them."""
    from flare_py_amd import fused

    for Cdim in (16, 96, 256):
        m = _lib.FlareMlpDesc()
        m.T, m.C, m.L, m.w_dtype = 16, Cdim, 1, _lib.DT_BF16
        assert _lib.load().flare_mlp_few(C.byref(m)) == fused._few(16, Cdim, 1) == 0
        assert fused._pair_info(torch.empty(16, Cdim), torch.nn.Linear(Cdim, Cdim), torch.nn.Linear(Cdim, Cdim), torch.bfloat16) is None


def _refused(rc, text, code=_lib.FLARE_EINVAL):
    assert rc == code and text in _lib.last_error(), (rc, _lib.last_error())


def test_causal_linear_bwd_validation():
    lib = _lib.load()
    d = _lib.FlareCausalLinearDesc()
    d.B, d.H, d.N, d.Dk, d.Dv, d.dtype = 1, 2, 256, 64, 64, _lib.DT_BF16
    d.q_stride = d.k_stride = d.v_stride = d.y_stride = _lib.I3(2 * 256 * 64, 256 * 64, 64)
    need = C.c_size_t(0)
    assert lib.flare_causal_linear_workspace_bytes(d, C.byref(need)) == _lib.FLARE_OK and need.value > 0
    fake = C.c_void_p(4096)

    def call(q=fake, gy=fake, gs=_lib.I3(2 * 256 * 64, 256 * 64, 64), ws=fake, have=need.value):
        return lib.flare_causal_linear_bwd(d, q, fake, fake, gy, gs, None, fake, fake, fake, ws, have, None)

    assert lib.flare_causal_linear_bwd(None, *([None] * 4), None, *([None] * 5), 0, None) == _lib.FLARE_EINVAL
    _refused(call(q=None), "must not be NULL")
    _refused(call(gy=None), "must not be NULL")
    _refused(call(gs=None), "must not be NULL")
    _refused(call(gs=_lib.I3(0, 0, 63)), "gy row stride")
    _refused(call(ws=None), "workspace", _lib.FLARE_EWORKSPACE)
    _refused(call(have=need.value - 1), "needed", _lib.FLARE_EWORKSPACE)
    _refused(call(ws=C.c_void_p(4098)), "4-byte")
    d.Dk = 129
    _refused(call(), "at most 128", _lib.FLARE_EUNSUPPORTED)
    d.Dk, d.v_stride = 64, _lib.I3(0, 0, 32)
    _refused(call(), "v row stride")


def test_triple_bwd_validation():
    lib = _lib.load()
    d = _lib.FlareTripleDesc()
    d.B, d.H, d.N, d.Dq, d.Dv, d.dtype = 1, 2, 256, 32, 32, _lib.DT_F16
    for n in ("q1", "q2", "k1", "k2", "v", "o"):
        setattr(d, n + "_stride", _lib.I3(2 * 256 * 32, 256 * 32, 32))
    need, fwd = C.c_size_t(0), C.c_size_t(0)
    _refused(lib.flare_triple_bwd_workspace_bytes(d, None), "bytes is NULL")
    assert lib.flare_triple_bwd_workspace_bytes(d, C.byref(need)) == _lib.FLARE_OK
    assert lib.flare_triple_workspace_bytes(d, C.byref(fwd)) == _lib.FLARE_OK and need.value > fwd.value > 0
    fake = C.c_void_p(4096)

    def call(null=None, ws=fake, have=need.value):
        ptrs = [None if i == null else fake for i in range(13)]
        ptrs[6] = None                                     # dstate may be missing
        return lib.flare_triple_bwd(d, *ptrs, ws, have, None)

    for i in range(13):
        if i != 6:
            _refused(call(null=i), "must not be NULL")
    _refused(call(ws=None), "workspace", _lib.FLARE_EWORKSPACE)
    _refused(call(have=need.value - 1), "needed", _lib.FLARE_EWORKSPACE)
    _refused(call(ws=C.c_void_p(4104)), "16-byte")
    d.normalize = 1
    _refused(call(), "neither a feature map nor the normaliser", _lib.FLARE_EUNSUPPORTED)
    d.normalize, d.feature_map = 0, 1
    _refused(call(), "neither a feature map nor the normaliser", _lib.FLARE_EUNSUPPORTED)
    d.feature_map, d.Dv = 0, 16
    _refused(call(), "Dq == Dv", _lib.FLARE_EUNSUPPORTED)
    d.Dq = d.Dv = 65
    _refused(call(), "at most 64", _lib.FLARE_EUNSUPPORTED)


def test_mlp_few_bwd_and_tiled_forward_validation():
    lib = _lib.load()
    m = _lib.FlareMlpDesc()
    m.T, m.C, m.L = 64, 128, 5
    m.x_dtype = m.y_dtype = m.res_dtype = m.w_dtype = _lib.DT_BF16
    m.norm, m.eps = 1, 1e-5
    m.x_stride = m.y_stride = m.res_stride = 128
    fake, odd = C.c_void_p(4096), C.c_void_p(4104)

    def call(x=fake, dy_a=fake, dy_b=fake, gamma=fake, add=0, a_in=fake, gb=fake):
        return lib.flare_mlp_few_bwd(m, x, dy_a, dy_b, fake, fake, fake, gamma, fake, add, fake, a_in, fake, gb, None)

    assert lib.flare_mlp_few_bwd(None, *([None] * 8), 0, *([None] * 5)) == _lib.FLARE_EUNSUPPORTED
    _refused(call(x=None), "must not be NULL")
    _refused(call(dy_a=odd), "16-byte")
    _refused(call(dy_b=odd), "dy_b")
    _refused(call(gamma=None), "norm")
    _refused(call(gb=None), "norm")
    _refused(call(a_in=None), "a_in and g_out")
    _refused(call(add=4), "unknown bits")
    for field, value in (("T", 12289), ("T", 0), ("L", 6), ("C", 96), ("flags", _lib.MLP_EXPAND)):
        keep = getattr(m, field)
        setattr(m, field, value)
        _refused(call(), "flare_mlp_few", _lib.FLARE_EUNSUPPORTED)
        setattr(m, field, keep)
    m.flags = _lib.MLP_W_TILED                                # the backward knows its operands' order without it
    _refused(call(), "flags must be 0", _lib.FLARE_EUNSUPPORTED)

    def forward():
        return lib.flare_mlp_fwd(m, fake, fake, fake, fake, fake, fake, fake, None)

    m.T = 12289
    _refused(forward(), "flare_mlp_few", _lib.FLARE_EUNSUPPORTED)
    m.T, m.L = 64, 6
    _refused(forward(), "flare_mlp_few", _lib.FLARE_EUNSUPPORTED)
    m.flags, m.L = _lib.MLP_W_TILED | _lib.MLP_EXPAND, 4
    _refused(forward(), "flare_mlp_few", _lib.FLARE_EUNSUPPORTED)
    m.flags, m.norm = _lib.MLP_W_TILED, 0
    _refused(lib.flare_mlp_io_fwd(m, 3, 1, fake, fake, 0, fake, fake, fake, None, None, None, fake, None), "flare_mlp_few", _lib.FLARE_EUNSUPPORTED)


def test_mlp_pack_validation():
    lib = _lib.load()
    fake, odd = C.c_void_p(4096), C.c_void_p(4104)

    def desc(**kw):
        d = _lib.FlareMlpPackDesc()
        d.L, d.C, d.w_dtype = 2, 64, _lib.DT_BF16
        for l in range(2):
            d.src[l], d.ld[l], d.rows[l] = 4096, 64, 64
        for k, v in kw.items():
            if isinstance(v, tuple):
                getattr(d, k)[v[0]] = v[1]
            else:
                setattr(d, k, v)
        return d

    def call(d, w=fake, img=None, img_t=None, bias=fake):
        return lib.flare_mlp_pack(d, w, img, img_t, bias, None)

    assert lib.flare_mlp_pack(None, *([None] * 5)) == _lib.FLARE_EINVAL
    _refused(call(desc(L=0)), "1 <= L")
    _refused(call(desc(L=_lib.MLP_PACK_MAX + 1)), "1 <= L")
    _refused(call(desc(w_dtype=_lib.DT_F32)), "w_dtype")
    _refused(call(desc(C=96)), "32, 64 and 128", _lib.FLARE_EUNSUPPORTED)
    _refused(call(desc(), w=None), "must not be NULL")
    _refused(call(desc(), bias=None), "must not be NULL")
    _refused(call(desc(), img=fake), "come together")
    _refused(call(desc(tiled=1), img=fake, img_t=fake), "come together")
    _refused(call(desc(), w=odd), "16-byte")
    _refused(call(desc(), img=fake, img_t=odd), "16-byte")
    _refused(call(desc(src=(1, None))), "src[1] is NULL")
    _refused(call(desc(rows=(0, 65))), "tile 0")
    _refused(call(desc(rows=(1, 0))), "tile 1")
    _refused(call(desc(ld=(1, 63))), "tile 1")
    _refused(call(desc(src_dtype=(0, 3))), "unknown dtype")
    _refused(call(desc(b_dtype=(1, -1))), "unknown dtype")


def test_mlp_wgrad_norm_validation():
    lib = _lib.load()
    m = _lib.FlareMlpDesc()
    m.T, m.C, m.L, m.w_dtype = 100, 64, 2, _lib.DT_BF16
    fake, odd = C.c_void_p(4096), C.c_void_p(4104)

    def call(part=fake, rows=7, gb=fake, a=fake):
        return lib.flare_mlp_wgrad_norm(m, a, 0, fake, 0, fake, None, None, None, part, rows, gb, None)

    _refused(call(a=None), "must not be NULL")
    _refused(call(part=None), "gb needs gb_part")
    _refused(call(rows=0), "gb needs gb_part")
    _refused(call(part=odd), "16-byte")
    _refused(call(gb=odd), "16-byte")


def test_row_pass_validation():
    lib = _lib.load()
    fake, odd, n = C.c_void_p(4096), C.c_void_p(4104), C.c_int32(0)
    assert lib.flare_rows_parts(1, 32, C.byref(n)) == _lib.FLARE_OK and n.value == 1
    assert lib.flare_rows_parts(1 << 40, 256, C.byref(n)) == _lib.FLARE_OK and 1 <= n.value <= 4096
    _refused(lib.flare_rows_parts(4, 32, None), "parts is NULL")
    _refused(lib.flare_rows_parts(0, 32, C.byref(n)), "T >= 1")
    _refused(lib.flare_rows_parts(4, 96, C.byref(n)), "only 32, 64, 128 and 256", _lib.FLARE_EUNSUPPORTED)

    def act(T=4, width=64, kind=0, ds=fake, t=fake, dt=fake, part=fake):
        return lib.flare_rows_act_bwd(T, width, kind, ds, t, dt, None, part, None, None)

    _refused(act(T=0), "T >= 1")
    _refused(act(width=48), "only 32", _lib.FLARE_EUNSUPPORTED)
    _refused(act(kind=2), "unknown activation")
    _refused(act(kind=-2), "unknown activation")
    _refused(act(ds=None), "required array is NULL")
    _refused(act(part=None), "required array is NULL")
    _refused(act(t=None), "must not be NULL with an activation")
    _refused(act(dt=None), "must not be NULL with an activation")
    _refused(act(ds=odd), "16-byte")

    def fwd(norm=1, eps=1e-5, x=fake, gamma=fake, stats=fake):
        return lib.flare_rows_norm_fwd(4, 64, norm, eps, x, gamma, None, fake, stats, None)

    _refused(fwd(norm=0), "unknown norm")
    _refused(fwd(eps=-1.0), "eps")
    _refused(fwd(eps=float("nan")), "eps")
    _refused(fwd(x=None), "required array is NULL")
    _refused(fwd(gamma=odd), "16-byte")
    _refused(fwd(stats=None), "required array is NULL")

    def bwd(norm=2, dy=fake, stats=fake, add=None, part=fake):
        return lib.flare_rows_norm_bwd(4, 64, norm, dy, fake, stats, None, add, fake, part, None, None)

    _refused(bwd(norm=3), "unknown norm")
    _refused(bwd(dy=None), "required array is NULL")
    _refused(bwd(stats=None), "required array is NULL")
    _refused(bwd(part=None), "required array is NULL")
    _refused(bwd(add=odd), "16-byte")


def test_block_end_pack_rows_and_partial_gradient_validation():
    """Argument errors of the few-token launches around a block are found on the host."""
    lib, fake, odd = _lib.load(), C.c_void_p(1 << 20), C.c_void_p((1 << 20) + 8)
    f, s = _lib.FlareMlpDesc(), _lib.FlareMlpDesc()
    for d in (f, s):
        d.T, d.C, d.L, d.w_dtype, d.x_stride, d.y_stride, d.res_stride = 16, 64, 1, 1, 64, 64, 64
        d.flags = _lib.MLP_W_TILED
    s.L, f.x_dtype = 3, 1

    def fwd(f_=f, s_=s, x=fake, res=fake, w1=fake, y=fake, gamma=None):
        return lib.flare_mlp_few_tail_fwd(f_, s_, x, res, w1, None, fake, None, gamma, None, None, y, None)

    assert fwd(None) == _lib.FLARE_EUNSUPPORTED and fwd(s_=None) == _lib.FLARE_EUNSUPPORTED
    assert fwd(x=odd) == _lib.FLARE_EINVAL and fwd(res=None) == _lib.FLARE_EINVAL and fwd(w1=None) == _lib.FLARE_EINVAL and fwd(y=odd) == _lib.FLARE_EINVAL
    for name, bad in (("L", 2), ("act_mask", 1), ("add_mask", 1), ("norm", 1), ("T", 17), ("C", 32), ("w_dtype", 2), ("x_dtype", 0), ("y_stride", 68), ("flags", 0)):
        old = getattr(f, name)
        setattr(f, name, bad)
        assert fwd() == _lib.FLARE_EUNSUPPORTED, name
        setattr(f, name, old)
    s.norm = 1
    assert fwd() == _lib.FLARE_EINVAL and "gamma" in _lib.last_error()
    s.norm = 0
    for d in (f, s):
        d.T = 16385
    assert fwd() == _lib.FLARE_EUNSUPPORTED

    for d in (f, s):
        d.T, d.flags = 16, 0

    def bwd(f_=f, s_=s, x1=fake, x=fake, wt1=fake, dx=fake, a=fake, dx1=fake):
        return lib.flare_mlp_few_tail_bwd(f_, s_, x1, fake, fake, fake, None, None, None, dx1, fake, fake, None, x, wt1, dx, a, fake, None)

    assert bwd(None) == _lib.FLARE_EUNSUPPORTED and bwd(s_=None) == _lib.FLARE_EUNSUPPORTED
    assert all(bwd(**{n: v}) == _lib.FLARE_EINVAL for n in ("x1", "x", "wt1", "dx", "a", "dx1") for v in (None, odd))
    f.flags = 3 << 8
    assert bwd() == _lib.FLARE_EINVAL
    f.flags = 2 << 8
    assert bwd() == _lib.FLARE_EINVAL and "row stride" in _lib.last_error()
    f.flags, s.T = 0, 17
    assert bwd() == _lib.FLARE_EUNSUPPORTED
    f.T = s.T = 16385
    assert bwd() == _lib.FLARE_EUNSUPPORTED

    p = _lib.FlareMlpPackDesc()
    p.L, p.C, p.w_dtype, p.tiled, p.src[0], p.rows[0], p.ld[0] = 1, 32, 1, 1, 1 << 20, 32, 32
    for rows in ((fake, 0, 4, 4, 0, fake), (fake, 2, 0, 4, 0, fake), (fake, 2, 8, 4, 0, fake), (fake, 2, 3, 6, 0, fake), (fake, 2, 4, 4, 3, fake),
                 (fake, 2, 4, 4, 0, None), (fake, 2, 4, 4, 0, odd)):
        assert lib.flare_mlp_pack_rows(p, fake, None, fake, fake, *rows, None) == _lib.FLARE_EINVAL

    m = _lib.FlareMixerDesc()
    m.B, m.H, m.N, m.M, m.D, m.dtype, m.scale = 1, 2, 100, 32, 16, 1, 1.0
    for n in ("q_stride", "k_stride", "v_stride", "y_stride"):
        setattr(m, n, _lib.I3(3200, 1600, 16))
    off, splits = C.c_size_t(0), C.c_int32(0)
    assert lib.flare_mixer_bwd_dq_parts(m, off, splits) == _lib.FLARE_OK and splits.value >= 1 and off.value % 16 == 0
    assert lib.flare_mixer_bwd_dq_parts(m, None, splits) == _lib.FLARE_EINVAL
    g = _lib.FlareMlpDesc()
    g.T, g.C, g.L, g.w_dtype = 100, 32, 1, 1

    def wgrad(m_=m, part=fake, n=1, cols=16, dq=fake):
        return lib.flare_mlp_wgrad_block(g, fake, 3200, fake, 3200, fake, None, None, None, None, None, 0, None, None, m_, part, n, cols, dq, None)

    assert wgrad(None) == _lib.FLARE_EINVAL and wgrad(part=odd) == _lib.FLARE_EINVAL and wgrad(dq=odd) == _lib.FLARE_EINVAL
    assert wgrad(n=0) == _lib.FLARE_EINVAL and all(wgrad(cols=c) == _lib.FLARE_EINVAL for c in (0, 6, 20))
    m.dtype = 0
    assert lib.flare_mixer_bwd_dq_parts(m, off, splits) == _lib.FLARE_EUNSUPPORTED
