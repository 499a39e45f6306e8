"""fp32 training of the token-wise layers through the row passes (rows.chain, rows.norm) against the same torch layers in fp64; the
error may not exceed what torch's own fp32 layers show by more than half (sums in another order), with 1e-7 for results that
torch happens to get exactly."""
import copy

import pytest
import torch
from torch import nn

import flare_py_amd as F
from flare_py_amd import modules, rows
from flare_py_amd.modules import ResidualMLP

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_size(monkeypatch):
    monkeypatch.setattr(rows, "MIN_ELEMS", 0)


def rel(a, b):
    return float((a.double() - b).norm() / (b.norm() + 1e-300))


def grads(fn, x, params, gy):
    y = fn(x)
    return [y.detach(), *torch.autograd.grad(y, [x, *params], gy)]


def hold(got, t32, ref):
    for i, (a, b, r) in enumerate(zip(got, t32, ref)):
        assert rel(a, r) <= 1.5 * rel(b, r) + 1e-7, (i, rel(a, r), rel(b, r))


@pytest.mark.parametrize("C,T,layers,act,ends", [(32, 4096, 3, "gelu", True), (64, 4097, 0, "silu", False), (128, 5003, 3, "gelu", True),
                                                 (256, 4099, 1, "silu", True), (128, 70001, -1, "gelu", True)])
def test_residual_mlp(dev, monkeypatch, C, T, layers, act, ends):
    torch.manual_seed(C)
    m = ResidualMLP(C, C, C, num_layers=layers, act=act, input_residual=ends, output_residual=ends).to(dev)
    if layers > 0:
        m.fcs[0].bias = None
    for p in m.parameters():
        p.data.mul_(2.0)
    x = (torch.randn(T, C, device=dev) * 3).requires_grad_(True)
    gy = torch.randn(T, C, device=dev)
    m64, x64 = copy.deepcopy(m).double(), x.detach().double().requires_grad_(True)
    ref = grads(m64, x64, list(m64.parameters()), gy.double())
    assert rows.chain_info(m, x) is not None
    got = grads(m, x, list(m.parameters()), gy)
    monkeypatch.setattr(modules, "_LONG_ROWS", 1 << 62)
    t32 = grads(m, x, list(m.parameters()), gy)
    monkeypatch.setattr(modules, "_LONG_ROWS", rows.LONG_ROWS)
    hold(got, t32, ref)
    again = grads(m, x, list(m.parameters()), gy)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("kind", [nn.LayerNorm, nn.RMSNorm])
@pytest.mark.parametrize("C,T", [(32, 4096), (64, 4105), (128, 4097), (256, 33001)])
def test_norm(dev, kind, C, T):
    torch.manual_seed(T)
    m = kind(C).to(dev)
    for p in m.parameters():
        p.data.add_(0.5 * torch.randn_like(p))
    x = (torch.randn(T, C, device=dev) * 2 + 1).requires_grad_(True)
    gy = torch.randn(T, C, device=dev)
    m64, x64 = copy.deepcopy(m).double(), x.detach().double().requires_grad_(True)
    m64.eps = m.eps if m.eps is not None else torch.finfo(torch.float32).eps
    ref = grads(m64, x64, list(m64.parameters()), gy.double())
    got = grads(lambda t: rows.norm(m, t), x, list(m.parameters()), gy)
    hold(got, grads(m, x, list(m.parameters()), gy), ref)


def test_strided_rows_frozen_parameters_and_hooks(dev):
    torch.manual_seed(0)
    m = ResidualMLP(64, 64, 64, num_layers=1, input_residual=True, output_residual=True).to(dev)
    wide = torch.randn(2, 3000, 67, device=dev)
    x = wide[..., 1:65]                                       # rows at a stride, off the 16-byte grid, no gradient asked for
    m.fc1.bias.requires_grad_(False)
    ref = m.double()(x.double())
    ref.sum().backward()
    want = [None if p.grad is None else p.grad.clone() for p in m.parameters()]
    m.float().zero_grad(set_to_none=True)
    y = m(x)
    assert rel(y.detach(), ref.detach()) <= 1e-6
    y.sum().backward()
    for p, r in zip(m.parameters(), want):
        assert (p.grad is None) == (r is None) and (r is None or rel(p.grad, r.double()) <= 1e-5)
    assert rows.chain_info(m, x) is not None
    seen = []
    h = m.act.register_forward_hook(lambda *a: seen.append(1))
    assert rows.chain_info(m, x) is None                      # a hook wants its layer called
    m(x)
    h.remove()
    assert seen
    m.fc2.weight.requires_grad_(False)
    assert rows.chain_info(m, x) is None
    with torch.no_grad():
        assert rows.chain_info(m, x) is None


@pytest.mark.parametrize("lra", [False, True])
def test_block_against_torch_layers(dev, monkeypatch, lra):
    from flare_py_amd import lra_modules

    torch.manual_seed(1)
    cls = lra_modules.FLAREBlock if lra else F.FLAREBlock
    kw = {"kv_proj_hidden_dim": 64, "ffn_hidden_dim": 64} if lra else {}
    m = cls(channel_dim=64, num_heads=4, num_latents=32, **kw).to(dev)
    x = torch.randn(2, 2500, 64, device=dev, requires_grad=True)
    gy = torch.randn(2, 2500, 64, device=dev)
    run = (lambda t: m(t)) if lra else (lambda t: m(t)[0])
    got = grads(run, x, list(m.parameters()), gy)
    monkeypatch.setattr(modules, "_LONG_ROWS", 1 << 62)
    t32 = grads(run, x, list(m.parameters()), gy)
    for a, b in zip(got, t32):
        assert rel(a, b.double()) <= 1e-5


def test_small_arrays_keep_the_torch_layers_outside_a_capture(dev, monkeypatch):
    monkeypatch.undo()
    m = ResidualMLP(64, 64, 64, num_layers=1, input_residual=True, output_residual=True).to(dev)
    assert rows.chain_info(m, torch.randn(8192, 64, device=dev)) is None
    assert rows.chain_info(m, torch.empty(rows.MIN_ELEMS // 64, 64, device=dev)) is not None


@pytest.mark.parametrize("C,elems", [(64, rows.MIN_ELEMS), (128, rows.MIN_ELEMS), (32, 6 << 20), (256, 6 << 20)])
def test_the_sizes_from_which_the_row_passes_run(dev, monkeypatch, C, elems):
    monkeypatch.undo()
    m = ResidualMLP(C, C, C, num_layers=1, input_residual=True, output_residual=True).to(dev)
    assert rows.chain_info(m, torch.empty(elems // C, C, device=dev)) is not None
    assert rows.chain_info(m, torch.empty(elems // C - 1, C, device=dev)) is None


def test_saved_tensors_may_come_back_in_another_memory_order(dev):
    """A saved-tensor hook owes the backward the values, not the strides."""
    torch.manual_seed(2)
    m, n = ResidualMLP(64, 64, 64, num_layers=1, input_residual=True, output_residual=True).to(dev), nn.LayerNorm(64).to(dev)
    x = torch.randn(4096, 64, device=dev, requires_grad=True)
    gy = torch.randn(4096, 64, device=dev)
    params = [*m.parameters(), *n.parameters()]
    run = lambda t: m(rows.norm(n, t))
    want = grads(run, x, params, gy)
    assert rows.chain_info(m, x) is not None
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.t().contiguous().t() if t.dim() == 2 else t):
        y = run(x)
    got = [y.detach(), *torch.autograd.grad(y, [x, *params], gy)]
    for a, b in zip(got, want):
        assert rel(a, b.double()) <= 1e-6


@pytest.mark.parametrize("lra", [False, True])
@pytest.mark.parametrize("how", ["forward replaced", "global hook"])
def test_replaced_forwards_and_global_hooks_are_called(dev, lra, how):
    from flare_py_amd import lra_modules

    cls = lra_modules.FLAREBlock if lra else F.FLAREBlock
    kw = {"kv_proj_hidden_dim": 64, "ffn_hidden_dim": 64} if lra else {}
    m = cls(channel_dim=64, num_heads=4, num_latents=32, **kw).to(dev)
    x = torch.randn(2, 2500, 64, device=dev, requires_grad=True)
    watched, seen = {m.norm1, m.norm2, m.mlp, m.mlp.act, m.att.k_proj.act}, set()
    handle = None
    if how == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, *a: seen.add(mod))
    else:
        for mod in watched:
            mod.forward = (lambda mod, f: lambda *a: (seen.add(mod), f(*a))[1])(mod, mod.forward)
    try:
        out = m(x)
    finally:
        if handle is not None:
            handle.remove()
    assert watched <= seen
    (out if lra else out[0]).sum().backward()
    assert bool(torch.isfinite(x.grad).all())


@pytest.mark.parametrize("norm", [1, 2])
@pytest.mark.parametrize("T,C", [(1, 32), (1000, 64), (4097, 256)])
def test_norm_backward_adds_another_gradient(dev, norm, T, C):
    """The C interface's optional gradient of x from another path (a residual's): added to dx, one rounding of the sum."""
    import ctypes

    from flare_py_amd import _lib

    lib = _lib.load()
    x, dy, add = (torch.randn(T, C, device=dev) for _ in range(3))
    gamma = torch.rand(C, device=dev) + 0.5
    y, stats = torch.empty_like(x), torch.empty(T, 2, device=dev)
    p = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.flare_rows_norm_fwd(T, C, norm, 1e-5, p(x), p(gamma), None, p(y), p(stats), st), "forward")
    part, gb = torch.empty(rows._parts(T, C), 2, C, device=dev), torch.empty(2, C, device=dev)
    dx = {}
    for a in (None, add):
        dx[a is add] = torch.empty_like(x)
        _lib.check(lib.flare_rows_norm_bwd(T, C, norm, p(dy), p(x), p(stats), p(gamma), p(a), p(dx[a is add]), p(part), p(gb), st), "backward")
    assert torch.equal(dx[True], dx[False] + add)
    xr = x.double().requires_grad_(True)
    yr = (nn.functional.layer_norm(xr, (C,), gamma.double(), None, 1e-5) if norm == 1 else nn.functional.rms_norm(xr, (C,), gamma.double(), 1e-5))
    (want,) = torch.autograd.grad(yr, xr, dy.double())
    assert rel(y, yr.detach()) <= 1e-6 and rel(dx[False], want) <= 1e-6


@pytest.mark.parametrize("act", [-1, 0, 1])
@pytest.mark.parametrize("T,C", [(1, 64), (15, 128), (64, 64), (65, 128), (177, 64), (4111, 128), (16384, 128), (16385, 64), (33000, 128), (40000, 64)])
def test_layer_backward_in_one_pass(dev, act, T, C):
    """flare_rows_layer_bwd against the layer's gradients in fp64: around a workgroup's least rows, the tile, the 16-row step and the
    first row counts that give every compute unit more than one tile.  Bound per result: 2e-6 of its norm, several times what sums of
    C (dx) or T (dw, db) products rounded in fp32 show."""
    import ctypes

    from flare_py_amd import _lib

    lib = _lib.load()
    torch.manual_seed(T)
    dy, x = torch.randn(T, C, device=dev), torch.randn(T, C, device=dev)
    w, b = torch.randn(C, C, device=dev) * C ** -0.5, torch.randn(C, device=dev)
    t = torch.nn.functional.linear(x, w, b) * 2
    n = ctypes.c_int32(0)
    _lib.check(lib.flare_rows_layer_bwd_parts(T, C, ctypes.byref(n)), "parts")
    assert 1 <= n.value <= 4096
    t64 = t.double().requires_grad_(True)
    f = (lambda v: v, lambda v: nn.functional.gelu(v, approximate="tanh"), nn.functional.silu)[act + 1]
    (dt,) = torch.autograd.grad(f(t64), t64, dy.double())
    p = lambda v: None if v is None else ctypes.c_void_p(v.data_ptr())
    for add, want_x, want_b in ((0, True, True), (1, True, False), (0, False, True)):
        guard = torch.full((T + 64, C), 7.0, device=dev)
        dx, dw, db = guard[:T] if want_x else None, torch.empty_like(w), torch.empty_like(b) if want_b else None
        pw, pb = torch.empty(n.value, C, C, device=dev), torch.empty(n.value, C, device=dev)
        _lib.check(lib.flare_rows_layer_bwd(T, C, act, add, p(dy), p(t) if act >= 0 else None, p(x), p(w), p(dx), p(pw), p(pb), p(dw), p(db),
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "flare_rows_layer_bwd")
        assert rel(dw, dt.t() @ x.double()) <= 2e-6
        if want_b:
            assert rel(db, dt.sum(0)) <= 2e-6 * max(1.0, float(dt.norm() / dt.sum(0).norm()))
        if want_x:
            assert rel(dx, dt @ w.double() + (dy.double() if add else 0)) <= 2e-6
            assert bool((guard[T:] == 7.0).all())


@pytest.mark.parametrize("T,C", [(1, 32), (4097, 64), (70001, 128)])
@pytest.mark.parametrize("act", [-1, 0])
def test_activation_and_sums_equal_the_torch_layers(dev, act, T, C):
    """Bit for bit, over every binade, signed zeros, subnormals, infinities and NaN; in place too."""
    import ctypes

    from flare_py_amd import _lib

    lib = _lib.load()
    torch.manual_seed(T)
    t = torch.randint(-2 ** 31, 2 ** 31 - 1, (T, C), device=dev, dtype=torch.int32).view(torch.float32)
    t[:, :16] = torch.randn(T, 16, device=dev) * 3
    t.view(-1)[:6] = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), 1e-40], device=dev)
    x, res = torch.randn(T, C, device=dev), torch.randn(T, C, device=dev)
    f = (lambda v: v) if act < 0 else (lambda v: nn.functional.gelu(v, approximate="tanh"))
    p = lambda v: None if v is None else ctypes.c_void_p(v.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for xx, rr in ((None, None), (x, None), (None, res), (x, res)):
        want = f(t)
        want = want if xx is None else xx + want
        want = want if rr is None else rr + want
        y, again = torch.empty_like(t), t.clone()
        _lib.check(lib.flare_rows_act_fwd(T, C, act, p(t), p(xx), p(rr), p(y), st), "flare_rows_act_fwd")
        _lib.check(lib.flare_rows_act_fwd(T, C, act, p(again), p(xx), p(rr), p(again), st), "flare_rows_act_fwd")
        for a in (y, again):
            assert torch.equal(torch.nan_to_num(a, nan=0.0, posinf=1e38, neginf=-1e38), torch.nan_to_num(want, nan=0.0, posinf=1e38, neginf=-1e38))
            assert torch.equal(a.isnan(), want.isnan())
    assert lib.flare_rows_act_fwd(T, C, 1, p(t), None, None, p(t), st) == _lib.FLARE_EUNSUPPORTED
