"""A FLAREBlock's inference forward through its plan (one call into the library) against the general path: the same launches on the same
operands, so the outputs are equal bit for bit; and what a plan was made from is looked at again by every call."""
import copy
import io

import pytest
import torch
from torch import nn

import flare_py_amd as F
from flare_py_amd import _lib, block_plan, functional

pytestmark = pytest.mark.gpu


def make(dev, C=64, H=4, M=64, **kw):
    torch.manual_seed(C + H + M)
    m = F.FLAREBlock(channel_dim=C, num_heads=H, num_latents=M, **kw).to(dev).eval()
    for l in m.modules():
        if isinstance(l, nn.Linear):
            l.reset_parameters()
    return m


def general(m, x, cd=torch.bfloat16, **kw):
    keep, block_plan.forward = block_plan.forward, lambda block, x: None
    try:
        with torch.no_grad(), torch.autocast("cuda", dtype=cd):
            return m(x, **kw)[0]
    finally:
        block_plan.forward = keep


def planned(m, x, cd=torch.bfloat16, used=True):
    """The second call of a block is the first one through a plan."""
    calls, lib = [], _lib.load()
    real = lib.flare_block_fwd
    lib.flare_block_fwd = lambda *a: (calls.append(1), real(*a))[1]
    try:
        with torch.no_grad(), torch.autocast("cuda", dtype=cd):
            m(x)
            del calls[:]
            y = m(x)[0]
    finally:
        lib.flare_block_fwd = real
    assert len(calls) == int(used)
    return y


# narrow heads (4, 8), every plain head dim, few and many tokens and either side of the line, expanding feed-forward, both norms
@pytest.mark.parametrize("C,H,M,B,N,kw", [(64, 8, 64, 1, 3973, {}), (32, 8, 32, 2, 77, {}), (128, 8, 128, 1, 1, {}), (64, 2, 96, 3, 1000, {"rmsnorm": True}),
                                          (128, 2, 64, 1, 12289, {"act": "silu"}), (64, 8, 64, 2, 8193, {}),
                                          (128, 8, 128, 1, 5000, {"num_layers_ffn": 0, "ffn_mlp_ratio": 4.0}),
                                          (64, 4, 64, 1, 20001, {"num_layers_ffn": 0, "ffn_mlp_ratio": 2.0, "num_layers_k_proj": 1}),
                                          (64, 4, 64, 1, 700, {"num_layers_ffn": -1, "num_layers_v_proj": 0})])
@pytest.mark.parametrize("cd,xd", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
def test_plan_equals_the_general_path(dev, C, H, M, B, N, kw, cd, xd):
    m = make(dev, C, H, M, **kw)
    x = torch.randn(B, N, C, device=dev).to(xd)
    want = general(m, x, cd)
    y = planned(m, x, cd)
    assert y.dtype == xd and torch.equal(y, want)
    x2 = torch.randn_like(x)                                    # other inputs of the shape, and the first ones again
    assert torch.equal(planned(m, x2, cd), general(m, x2, cd)) and torch.equal(planned(m, x, cd), want)


def test_a_plan_follows_its_module(dev):
    m = make(dev)
    x = torch.randn(2, 500, 64, device=dev)
    planned(m, x)

    def same():
        assert torch.equal(planned(m, x), general(m, x))

    before = planned(m, x)
    for p in (m.mlp.fc1.weight, m.att.k_proj.fc2.bias, m.att.latent_q, m.norm2.weight):
        with torch.no_grad():
            p.mul_(1.5).add_(0.01)
        same()
    m.att.v_proj.fcs[0] = nn.Linear(64, 64).to(dev)
    same()
    m.mlp.fc2.bias = nn.Parameter(torch.randn(64, device=dev))
    same()
    m.norm1.weight.data = torch.rand(64, device=dev)
    same()
    m.att.attn_scale, m.norm1.eps = 0.5, 1e-2
    same()
    m.mlp.act = nn.SiLU()
    same()
    assert not torch.equal(before, planned(m, x))
    with functional.mixer_flags(_lib.FLAG_MFMA16):
        same()
    c = copy.deepcopy(m)
    assert not c._flare_plans and torch.equal(planned(c, x), planned(m, x))
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    assert torch.equal(planned(torch.load(buf, weights_only=False), x), planned(m, x))
    for n in range(1, 40):                                       # plans are bounded
        planned(m, x[:, :n].contiguous())
    assert len(m._flare_plans) <= block_plan._MAX_SHAPES


@pytest.mark.parametrize("how", ["data", "parameter"])
@pytest.mark.parametrize("what", ["layer", "latents"])
def test_replaced_weights_reach_the_plans_of_every_shape(dev, how, what):
    """Weights replaced between calls on two shapes: an earlier one's memory comes back under a later one, at the same version."""
    m = make(dev)
    a, b = torch.randn(2, 500, 64, device=dev), torch.randn(1, 700, 64, device=dev)
    owner, name = (m.mlp.fc1, "weight") if what == "layer" else (m.att, "latent_q")
    w0 = getattr(owner, name).detach().clone()

    def value(i):
        return w0 * (1.0 + 0.125 * i)

    def replace(i):
        if how == "data":
            getattr(owner, name).data = value(i)
        else:
            setattr(owner, name, nn.Parameter(value(i)))

    want = []
    for i in range(24):
        n = make(dev)
        (n.mlp.fc1.weight if what == "layer" else n.att.latent_q).data.copy_(value(i))
        want.append((general(n, a), general(n, b)))
    planned(m, a)
    for i in range(0, 24, 3):
        replace(i)
        assert torch.equal(planned(m, b), want[i][1]), i
        replace(i + 1)
        assert torch.equal(planned(m, b), want[i + 1][1]), i
        replace(i + 2)
        assert torch.equal(planned(m, a), want[i + 2][0]), i
    m.cpu()
    assert "_flare_plans" not in m.__dict__


def test_shapes_that_a_block_meets_once(dev):
    """Each of them takes a plan, right away and after others took its place, and equals the general path."""
    m = make(dev)
    xs = [torch.randn(1, 100 + 7 * n, 64, device=dev) for n in range(block_plan._MAX_SHAPES + 3)] + [torch.randn(1, 13000, 64, device=dev)]
    planned(m, xs[0])
    calls, lib = [], _lib.load()
    real = lib.flare_block_fwd
    lib.flare_block_fwd = lambda *a: (calls.append(1), real(*a))[1]
    try:
        for x in (*xs, *xs):
            n = len(calls)
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
                y = m(x)[0]
            assert len(calls) == n + 1 and len(m._flare_plans) <= block_plan._MAX_SHAPES
            assert torch.equal(y, general(m, x))
    finally:
        lib.flare_block_fwd = real


def test_calls_that_keep_the_general_path(dev):
    m = make(dev)
    x = torch.randn(2, 300, 64, device=dev)
    wide = torch.randn(2, 300, 72, device=dev)
    off = torch.randn(2 * 300 * 64 + 1, device=dev)[1:].view(2, 300, 64)
    assert torch.equal(planned(m, wide[..., :64], used=False), general(m, wide[..., :64].contiguous()))
    assert torch.equal(planned(m, off, used=False), general(m, off.clone()))
    seen = []
    h = m.att.register_forward_hook(lambda *a: seen.append(1))
    planned(m, x, used=False)
    h.remove()
    assert len(seen) == 2
    m.att.forward = (lambda f: lambda *a, **k: (seen.append(1), f(*a, **k))[1])(m.att.forward)
    planned(m, x, used=False)
    del m.att.__dict__["forward"]
    assert len(seen) == 4
    torch.nn.utils.parametrizations.weight_norm(m.mlp.fc1)
    planned(m, x, used=False)
    for kw in ({"M": 40}, {"C": 64, "H": 64 // 2}, {"qk_norm": True}):            # dead latents, head dim 2, norms between
        planned(make(dev, **kw), x, used=False)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = make(dev)(x)[0]
    assert y.requires_grad
    half = make(dev).bfloat16()
    with torch.no_grad():
        half(x.bfloat16())
        half(x.bfloat16())
    assert not half.__dict__.get("_flare_plans")


@pytest.mark.parametrize("how", [None, nn.Identity()])
@pytest.mark.parametrize("grad", [False, True])
def test_a_block_without_norms(dev, how, grad):
    m = make(dev)
    x = torch.randn(2, 300, 64, device=dev)
    planned(m, x)
    m.norm1 = m.norm2 = how
    if grad:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = m(x)[0].detach()
        assert torch.equal(y, general(m, x))
    else:
        assert torch.equal(planned(m, x, used=False), general(m, x))


@pytest.mark.parametrize("name", ["weight", "bias"])
def test_a_parametrised_layer_keeps_the_general_path(dev, name):
    """Its weight or bias is another tensor at every access: a plan could serve one call only."""
    m = make(dev)
    torch.nn.utils.parametrize.register_parametrization(m.mlp.fc1, name, nn.Identity())
    x = torch.randn(2, 300, 64, device=dev)
    assert torch.equal(planned(m, x, used=False), general(m, x))


@pytest.mark.parametrize("warm_ups", [1, 2, 3])
@pytest.mark.parametrize("N", [300, 20000])
def test_a_recorded_forward_leaves_eager_calls_their_weights(dev, N, warm_ups):
    """What a recording packs is written by its replays alone."""
    m = make(dev)
    x = torch.randn(1, N, 64, device=dev)
    want = general(make(dev), x)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(warm_ups):
                m(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m(x)[0]
        assert torch.equal(m(x)[0], want) and torch.equal(m(x)[0], want)
        for _ in range(3):
            y.zero_()
            graph.replay()
            assert torch.equal(y, want) and torch.equal(m(x)[0], want)
