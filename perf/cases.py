"""What the performance of this package is measured on: the calls its users make, over the sizes they make them at.

Twelve listed cases and a generator of further ones over the same ranges:

    mixer     flare_multihead_mixer, forward alone or forward and backward (operator API)
    block     one FLAREBlock forward over batches of point clouds, under autocast (inference)
    model     a whole FLAREModel forward, eager, under autocast (inference)
    layer     one FLARE layer forward and backward over a long point cloud, under autocast
    graphed   a FLAREModel training step on a small mesh through GraphedTrainStep
    sequence  one sequence-model FLARE block, forward and backward, over a padded batch
    prefill   causal FLARE over a prompt
    decode    one recurrent step of causal FLARE on a state advanced in place
    linear    causal linear attention, forward alone or forward and backward
    triple    triple attention, forward alone or forward and backward

Module gradients come back as the one flat bucket that a data-parallel program reduces or a program with gradient
clipping takes the norm of, parameters in module order.
"""
import math

import torch

import flare_py_amd as F
from flare_py_amd import lra_modules

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}


# ---- the cases ------------------------------------------------------------------------------------------------------
def listed():
    return [
        # A small point cloud through the bare operator in fp32 (the reference's default precision): launch latency counts.
        {"name": "mixer_small_f32", "kind": "mixer", "dtype": "f32", "B": 1, "H": 8, "N": 4096, "M": 64, "D": 16, "grad": False, "mask": False},
        # The million-token forward the package is built around (bench.py's default workload).
        {"name": "mixer_1m_bf16", "kind": "mixer", "dtype": "bf16", "B": 1, "H": 8, "N": 1048576, "M": 256, "D": 32, "grad": False, "mask": False},
        # Training through the operator at the head dim of the 128-channel models, two clouds of a length nobody rounded.
        {"name": "mixer_train_bf16", "kind": "mixer", "dtype": "bf16", "B": 2, "H": 8, "N": 100003, "M": 128, "D": 16, "grad": True, "mask": False},
        # Inference over four clouds with the 4x feed-forward (bench.py --workload block, without its lift).
        {"name": "block_bf16", "kind": "block", "dtype": "bf16", "B": 4, "N": 65536, "C": 128, "H": 8, "M": 128, "ffn": 4},
        # The default model geometry (64 channels, 8 heads of 8) on one small mesh, as a script calls it.
        {"name": "model_small_bf16", "kind": "model", "dtype": "bf16", "B": 1, "N": 3973, "C": 64, "H": 8, "M": 64, "blocks": 8},
        # The time/memory benchmark of one layer at a million points (bench.py --workload layer), M = 512.
        {"name": "layer_1m_f16", "kind": "layer", "dtype": "f16", "B": 1, "N": 1000000, "C": 128, "H": 8, "M": 512},
        # A training step of the 8-block model on a small mesh, replayed (bench.py --workload model).
        {"name": "model_train_bf16", "kind": "graphed", "dtype": "bf16", "B": 1, "N": 4096, "C": 128, "H": 8, "M": 128, "blocks": 8},
        # The sequence benchmark's block at its own precision, batch and a padded length (bench.py --workload lra).
        {"name": "sequence_train_f32", "kind": "sequence", "dtype": "f32", "B": 32, "N": 2048, "C": 128, "H": 8, "M": 128},
        # A prompt of 8192 tokens (bench.py --workload causal), and then one token at a time.
        {"name": "prefill_bf16", "kind": "prefill", "dtype": "bf16", "B": 8, "H": 16, "N": 8192, "M": 128, "D": 64},
        {"name": "decode_bf16", "kind": "decode", "dtype": "bf16", "B": 8, "H": 16, "N": 1, "M": 128, "D": 64},
        # Causal linear attention in training at the usual head width.
        {"name": "linear_train_bf16", "kind": "linear", "dtype": "bf16", "B": 4, "H": 8, "N": 16384, "Dk": 64, "Dv": 64, "grad": True},
        # Triple attention forward and backward as the reference's own kernel benchmark runs it (fp16, D = 32).
        {"name": "triple_train_f16", "kind": "triple", "dtype": "f16", "B": 1, "H": 8, "N": 32768, "D": 32, "grad": True},
    ]


def _size(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm; as often odd as not."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, lo, hi, B):
    """A token count for a batch of B such that B * N lies between lo and hi."""
    return max(1, _size(rng, lo, hi) // B)


def draw(rng):
    kind = rng.choice(["mixer", "mixer", "block", "model", "layer", "graphed", "sequence", "sequence", "prefill", "decode", "linear", "triple"])
    half = rng.choice(["bf16", "bf16", "f16"])
    c = {"kind": kind, "dtype": half}
    if kind == "mixer":
        c["dtype"] = rng.choice(["bf16", "bf16", "f16", "f32"])
        c["B"], c["H"], c["M"], c["D"] = rng.choice([1, 1, 2, 4, 8]), rng.choice([4, 8]), rng.choice([32, 64, 128, 256]), rng.choice([8, 16, 32, 64])
        top = 600_000 if c["dtype"] != "f32" else 60_000
        c["N"] = _rows(rng, 2_000, top * 16 // max(16, c["D"]), c["B"])
        c["grad"], c["mask"] = rng.random() < 0.5, c["B"] > 1 and rng.random() < 0.5
    elif kind == "block":
        c["B"], c["C"], c["H"], c["M"], c["ffn"] = rng.choice([1, 2, 4]), rng.choice([64, 128]), 8, rng.choice([64, 128, 256]), rng.choice([1, 4])
        c["N"] = _rows(rng, 4_000, 300_000, c["B"])
    elif kind == "model":
        c["B"], c["C"], c["H"], c["M"], c["blocks"] = rng.choice([1, 1, 2]), rng.choice([64, 128]), 8, rng.choice([64, 128]), rng.choice([4, 8])
        c["N"] = _rows(rng, 1_000, 40_000, c["B"])
    elif kind == "layer":
        c["B"], c["C"], c["H"], c["M"] = 1, rng.choice([64, 128]), 8, rng.choice([128, 256, 512])
        c["N"] = _size(rng, 10_000, 500_000)
    elif kind == "graphed":
        c["dtype"] = "bf16"
        c["B"], c["C"], c["H"], c["M"], c["blocks"] = rng.choice([1, 2]), rng.choice([64, 128]), 8, rng.choice([64, 128]), rng.choice([4, 8])
        c["N"] = _rows(rng, 1_000, 20_000, c["B"])
    elif kind == "sequence":
        c["dtype"] = rng.choice(["f32", "f32", half])
        c["B"], c["C"], c["H"], c["M"] = rng.choice([8, 16, 32]), rng.choice([64, 128]), 8, rng.choice([32, 64, 128])
        c["N"] = _rows(rng, 8_000, 130_000, c["B"])
    elif kind == "prefill":
        c["B"], c["H"], c["D"] = rng.choice([1, 2, 4, 8]), rng.choice([8, 16]), rng.choice([32, 64])
        c["M"] = rng.choice([64, 128, 256]) if c["D"] == 32 else rng.choice([64, 128])
        c["N"] = _rows(rng, 1_000, 60_000, c["B"])
    elif kind == "decode":
        c["B"], c["H"], c["D"], c["N"] = rng.choice([1, 3, 8, 16]), rng.choice([8, 12, 16]), rng.choice([32, 64]), 1
        c["M"] = rng.choice([128, 256]) if c["D"] == 32 else 128
    elif kind == "linear":
        c["dtype"] = rng.choice(["bf16", "f16", "f32"])
        c["B"], c["H"], c["Dk"] = rng.choice([1, 2, 4]), rng.choice([4, 8]), rng.choice([64, 64, 128]) if c["dtype"] != "f32" else 64
        c["Dv"] = c["Dk"]
        c["N"] = _rows(rng, 2_000, 100_000, c["B"])
        c["grad"] = rng.random() < 0.6
    else:
        c["dtype"] = rng.choice(["bf16", "f16", "f16"])
        c["B"], c["H"], c["D"] = rng.choice([1, 2, 4]), rng.choice([4, 8]), rng.choice([16, 32])
        c["N"] = _rows(rng, 1_000, 65_536, c["B"])
        c["grad"] = rng.random() < 0.6
    return c


# ---- what a program has in hand before the call ---------------------------------------------------------------------
def _lengths_mask(B, N, g, dev):
    """Right-padded batch: lengths between a quarter of N and N, at least one of them full."""
    n = torch.randint(max(1, N // 4), N + 1, (B,), generator=g, device=dev)
    n[0] = N
    return torch.arange(N, device=dev)[None, :] < n[:, None]


def _rand_points(c, g, dev):
    """Coordinates in the unit square and one field value."""
    return torch.cat([torch.rand(c["B"], c["N"], 2, generator=g, device=dev), torch.randn(c["B"], c["N"], 1, generator=g, device=dev)], dim=-1)


def _mse(y, target):
    return torch.nn.functional.mse_loss(y.float(), target)


LOSS_SCALE = {"f16": 65536.0}                      # where torch's GradScaler starts; fp16 gradients underflow without it


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    kind = case["kind"]
    s = {"case": case}

    def randn(*shape, std=1.0, dtype=None):
        return (torch.randn(*shape, generator=g, device=dev) * std).to(dt if dtype is None else dtype)

    if kind in ("mixer", "prefill", "decode"):
        B, H, N, M, D = (case[n] for n in "BHNMD")
    if kind == "mixer":
        s["q"], s["k"], s["v"] = randn(H, M, D, std=D ** -0.5), randn(B, H, N, D), randn(B, H, N, D)
        s["mask"] = _lengths_mask(B, N, g, dev) if case["mask"] else None
        if case["grad"]:
            s["gy"] = randn(B, H, N, D)
            for n in "qkv":
                s[n].requires_grad_(True)
    elif kind in ("prefill", "decode"):
        std = D ** -0.25
        s["q"], s["k"], s["v"] = randn(H, M, D, std=std), randn(B, H, N, D, std=std), randn(B, H, N, D, std=std)
        if kind == "decode":                       # the state behind a prompt, and the buffers a decoding loop keeps
            kp, vp = randn(B, H, 512, D, std=std), randn(B, H, 512, D, std=std)
            _, s["state"] = F.flare_causal_prefill(s["q"], kp, vp)
            s["ws"], s["y"] = F.causal_workspace(s["q"], s["k"]), torch.empty_like(s["k"])
    elif kind == "linear":
        B, H, N = (case[n] for n in "BHN")
        s["q"], s["k"], s["v"] = randn(B, H, N, case["Dk"]), randn(B, H, N, case["Dk"]), randn(B, H, N, case["Dv"])
        if case["grad"]:
            s["gy"] = randn(B, H, N, case["Dv"])
            for n in "qkv":
                s[n].requires_grad_(True)
    elif kind == "triple":
        B, H, N, D = (case[n] for n in "BHND")
        qk = [randn(B, H, N, D, std=D ** -0.5) for _ in range(4)]
        if case["grad"]:                           # the layer applies its feature map first and differentiates through it
            qk = [torch.nn.functional.elu(t) + 1 for t in qk]
            s["gy"] = randn(B, H, N, D)
        s["in"] = [*qk, randn(B, H, N, D)]
        if case["grad"]:
            for t in s["in"]:
                t.requires_grad_(True)
    else:
        torch.manual_seed(seed)                    # weights as a fresh module has them
        C, H, M = case["C"], case["H"], case["M"]
        if kind == "block":
            ffn = {"num_layers_ffn": 0, "ffn_mlp_ratio": 4.0} if case["ffn"] == 4 else {}
            m = F.FLAREBlock(channel_dim=C, num_heads=H, num_latents=M, **ffn)
            s["x"] = randn(case["B"], case["N"], C, dtype=torch.float32)
        elif kind in ("model", "graphed"):
            m = F.FLAREModel(in_dim=3, out_dim=1, channel_dim=C, num_blocks=case["blocks"], num_heads=H, num_latents=M)
            if kind == "model":                    # inference meets weights that have left the near-zero initialisation
                for layer in m.modules():
                    if isinstance(layer, torch.nn.Linear):
                        layer.reset_parameters()
            s["x"] = _rand_points(case, g, dev)
            s["target"] = randn(case["B"], case["N"], 1, dtype=torch.float32)
        elif kind == "layer":
            m = F.FLARE(channel_dim=C, num_heads=H, num_latents=M)
            s["x"] = randn(case["B"], case["N"], C, dtype=torch.float32).requires_grad_(True)
            s["target"] = randn(case["B"], case["N"], C, dtype=torch.float32)
        else:
            m = lra_modules.FLAREBlock(channel_dim=C, num_heads=H, num_latents=M, num_layers_kv_proj=3, num_layers_ffn=3,
                                       kv_proj_hidden_dim=C, ffn_hidden_dim=C)
            s["x"] = randn(case["B"], case["N"], C, dtype=torch.float32).requires_grad_(True)
            s["mask"] = _lengths_mask(case["B"], case["N"], g, dev)
            s["gy"] = randn(case["B"], case["N"], C, dtype=torch.float32)      # what the blocks above send back
        s["m"] = m.to(dev).train(kind in ("layer", "graphed", "sequence"))
        s["params"] = list(m.parameters())
        if kind == "graphed":
            s["step"] = F.GraphedTrainStep(m, _mse, autocast_dtype=dt)
            s["step"](s["x"], s["target"])         # the capture
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------
def _autocast(case):
    dt = DTYPES[case["dtype"]]
    return torch.autocast("cuda", dtype=dt, enabled=dt != torch.float32)


def _bucket(params):
    return torch.cat([p.grad.reshape(-1) for p in params])


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mixer":
        if not case["grad"]:
            return F.flare_multihead_mixer(s["q"], s["k"], s["v"], key_mask=s["mask"])
        y = F.flare_multihead_mixer(s["q"], s["k"], s["v"], key_mask=s["mask"])
        return (y, *torch.autograd.grad(y, (s["q"], s["k"], s["v"]), s["gy"]))
    if kind == "prefill":
        return F.flare_causal_prefill(s["q"], s["k"], s["v"])
    if kind == "decode":
        return F.flare_causal_decode_step(s["q"], s["k"], s["v"], s["state"], inplace=True, workspace=s["ws"], out=s["y"])
    if kind == "linear":
        y = F.CausalLinear.apply(s["q"], s["k"], s["v"])
        return (y, *torch.autograd.grad(y, (s["q"], s["k"], s["v"]), s["gy"])) if case["grad"] else y
    if kind == "triple":
        if not case["grad"]:
            return F.triple_attention(*s["in"], feature_map="elu", normalize=True)
        state, y = F.TripleAttentionFunction.apply(*s["in"])
        return (state, y, *torch.autograd.grad(y, s["in"], s["gy"]))
    if kind == "graphed":
        loss = s["step"](s["x"], s["target"])
        return loss, _bucket(s["params"])
    m = s["m"]
    if kind in ("block", "model"):
        with torch.no_grad(), _autocast(case):
            y = m(s["x"])
        return y[0] if kind == "block" else y
    m.zero_grad(set_to_none=True)
    s["x"].grad = None
    with _autocast(case):
        if kind == "layer":
            loss = torch.nn.functional.mse_loss(m(s["x"])[0], s["target"])
        else:
            y = m(s["x"], s["mask"])
    if kind == "layer":
        (loss * LOSS_SCALE.get(case["dtype"], 1.0)).backward()
        return loss, s["x"].grad, _bucket(s["params"])
    y.backward(s["gy"])
    return y, s["x"].grad, _bucket(s["params"])


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    B, N, H = case["B"], case["N"], case["H"]
    if kind == "mixer":                            # q, k, v in, y out; with gradients dy in and dq, dk, dv out; 4 products, 10 more behind
        M, D = case["M"], case["D"]
        rows = B * H * N * D * e
        if case["grad"]:
            return {"bytes": 6 * rows + 2 * H * M * D * e, "flops": 14 * 2 * B * H * N * M * D}
        return {"bytes": 3 * rows + H * M * D * e, "flops": 4 * 2 * B * H * N * M * D}
    if kind in ("prefill", "decode"):              # q, k, v in, y out, the state out (and in); scores, state update, readout
        M, D = case["M"], case["D"]
        state = B * H * M * (D + 2) * 4
        return {"bytes": 3 * B * H * N * D * e + H * M * D * e + (2 if kind == "decode" else 1) * state, "flops": 3 * 2 * B * H * N * M * D}
    if kind == "linear":                           # the state's update and its product with q, each way
        Dk, Dv = case["Dk"], case["Dv"]
        fwd = {"bytes": B * H * N * 2 * (Dk + Dv) * e, "flops": 2 * 2 * B * H * N * Dk * Dv}
        if not case["grad"]:
            return fwd
        return {"bytes": 2 * fwd["bytes"], "flops": 4 * fwd["flops"]}
    if kind == "triple":                           # q1, q2, k1, k2, v in, out and the state out; each way two contractions with D^3 per token
        D = case["D"]
        rows, state = B * H * N * D * e, B * H * D ** 3 * 4
        if not case["grad"]:
            return {"bytes": 6 * rows + state, "flops": 2 * 2 * B * H * N * D ** 3}
        return {"bytes": 12 * rows + state, "flops": 8 * 2 * B * H * N * D ** 3}
    C, M = case["C"], case["M"]
    T = B * N
    linear, mixer = 2 * T * C * C, 8 * T * C * M   # one C x C layer, the mixer's four products
    if kind == "layer":                            # 11 layers, three products each; x, target in, dx out
        par = 11 * (C * C + C) + C * M
        return {"bytes": 3 * T * C * 4 + 2 * par * 4, "flops": 3 * 11 * linear + 3.5 * mixer}
    if kind == "sequence":                         # 16 layers; x, dy in, y, dx out
        par = 16 * (C * C + C) + C * M + 4 * C
        return {"bytes": 4 * T * C * 4 + 2 * par * 4, "flops": 3 * 16 * linear + 3.5 * mixer}
    if kind == "block":                            # x in, y out
        ffn = 8 if case["ffn"] == 4 else 5
        par = (11 + ffn) * (C * C + C) + C * M + 4 * C
        return {"bytes": 2 * T * C * 4 + par * 4, "flops": (11 + ffn) * linear + mixer}
    par = case["blocks"] * (16 * (C * C + C) + C * M + 4 * C) + 6 * C * C
    flops = case["blocks"] * (16 * linear + mixer) + 6 * linear
    if kind == "model":                            # points in, one value a point out
        return {"bytes": T * 4 * 4 + par * 4, "flops": flops}
    return {"bytes": T * 4 * 4 + 2 * par * 4, "flops": 3 * flops}      # graphed: the parameters in, their gradients out


# About four times the error of each path against the same path in fp32 (16-bit types), or against fp64 (fp32), largest output:
# mixer 2.6e-3 forward, 5.7e-3 with gradients (dq), fp32 2e-7 and 7e-7; prefill and decode 2.5e-3 (the state's sums); linear
# 2.4e-3 bf16, 2.9e-4 f16, 7e-7 fp32; triple 1.7e-3, 4e-4; block 1.6e-3, 1.7e-4; model 6.4e-3, 4.5e-4; layer 2.8e-3, 4.5e-4;
# sequence 3.6e-3, 6e-4, fp32 6e-7; graphed 7e-3, where single elements of the bucket are off by half the bucket's rms
# (gradients that nearly cancel, next to the large ones of the last layers).
_REL = {
    "mixer": {"bf16": 0.01, "f16": 0.01, "f32": 1e-6},
    "mixer+grad": {"bf16": 0.022, "f16": 0.022, "f32": 3e-6},
    "prefill": {"bf16": 0.01, "f16": 0.01},
    "decode": {"bf16": 0.01, "f16": 0.01},
    "linear": {"bf16": 0.01, "f16": 0.0012, "f32": 3e-6},
    "linear+grad": {"bf16": 0.01, "f16": 0.0012, "f32": 3e-6},
    "triple": {"bf16": 0.008, "f16": 0.0016},
    "triple+grad": {"bf16": 0.008, "f16": 0.0016},
    "block": {"bf16": 0.0065, "f16": 0.0007},
    "model": {"bf16": 0.026, "f16": 0.002},
    "layer": {"bf16": 0.012, "f16": 0.002},
    "graphed": {"bf16": 0.028},
    "sequence": {"bf16": 0.015, "f16": 0.0025, "f32": 3e-6},
}


def tolerance(case):
    """Largest relative error another correct implementation at the same precision would show."""
    rel = _REL[case["kind"] + ("+grad" if case.get("grad") else "")][case["dtype"]]
    return {"rel": rel, "max": 0.99} if case["kind"] == "graphed" else {"rel": rel}
