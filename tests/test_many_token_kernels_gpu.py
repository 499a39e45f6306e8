"""The many-token kernels of the fused MLP chain (mlp_mfma.hip, mlp_bwd_mfma.hip).

Launches of up to 12,288 tokens (C = 128) or 16,384 (C = 32, 64) take the few-token kernels, the sizes of most tests of the chain
among them.  Here those tests run again with that limit lowered to zero, so that the kernels behind it see the same edges (a ragged
last tile, one token, every depth, norm, activation and type), and at the first token counts beyond the real limit, where the
chain's instances with one tile per wave end (32,768) and the next one.  Bounds and oracles are those of the tests themselves.
"""
import pytest
import test_fused_gpu as forward
import test_fused_train_gpu as train
import torch
from torch import nn

from flare_py_amd import fused
from oracle import flare_oracle as O

pytestmark = pytest.mark.gpu


def _none_few(*args):
    raise AssertionError("a few-token launch")


@pytest.fixture
def many(monkeypatch):
    monkeypatch.setattr(fused, "_FEW_TOKENS", dict.fromkeys(fused._FEW_TOKENS, 0))
    monkeypatch.setattr(fused, "_packed_few", _none_few)


@pytest.mark.parametrize("C", [32, 64, 128])
@pytest.mark.parametrize("n,ir,orr,act", [(3, True, True, "gelu"), (0, False, True, "silu"), (1, True, False, "gelu"),
                                          (-1, True, True, "gelu"), (6, True, True, "silu")])
def test_forward_stacks(dev, many, C, n, ir, orr, act):
    forward.test_mlp_stack_vs_oracle(dev, C, n, ir, orr, act)


@pytest.mark.parametrize("norm_kind", ["layer", "rms"])
@pytest.mark.parametrize("xdt,odt,cd", [(torch.float32, torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.bfloat16, torch.bfloat16),
                                        (torch.float32, torch.float32, torch.float16), (torch.float16, torch.float16, torch.float16)])
def test_norm_residual_dtypes_and_ragged_rows(dev, many, norm_kind, xdt, odt, cd):
    forward.test_norm_residual_dtypes_and_ragged_rows(dev, norm_kind, xdt, odt, cd)


@pytest.mark.parametrize("C,hd", [(64, 8), (32, 4), (128, 8), (32, 8)])
def test_head_padded_rows_and_strided_rows(dev, many, C, hd):
    forward.test_head_padded_rows(dev, C, hd)
    forward.test_single_linear_with_residual_and_strided_rows(dev)


@pytest.mark.parametrize("C,T", [(128, 12289), (64, 16385), (32, 16385), (128, 32768), (64, 32768), (32, 32768), (128, 32769), (64, 32769)])
def test_forward_at_the_ends_of_the_instances(dev, monkeypatch, C, T):
    monkeypatch.setattr(fused, "_packed_few", _none_few)
    m = forward.make_mlp(C, 3, True, True, "gelu", dev, seed=T)
    norm = nn.LayerNorm(C).to(dev)
    nn.init.normal_(norm.weight, 1.0, 0.3)
    nn.init.normal_(norm.bias, 0.0, 0.3)
    x = torch.randn(T, C, device=dev) * 1.5 + 0.3
    with torch.no_grad():
        y = fused.fused_mlp(x, m, torch.bfloat16, norm=norm, res=x)
    ref = forward.oracle_of(m, x, torch.bfloat16, norm, x)
    assert O.rel_l2(y, ref) <= 2e-2
    assert O.rel_l2(y[-64:], ref[-64:]) <= 2e-2


@pytest.mark.parametrize("C,num_layers,T,norm_kind,dtype,act", [
    (64, 3, 1000, "ln", torch.bfloat16, "gelu"), (128, 3, 700, "ln", torch.bfloat16, "gelu"), (32, 3, 333, "rms", torch.bfloat16, "gelu"),
    (128, -1, 500, None, torch.bfloat16, "gelu"), (64, 6, 129, "ln", torch.float16, "silu"), (64, 0, 777, "ln", torch.bfloat16, "gelu"),
    (32, 6, 17, None, torch.bfloat16, "silu"), (32, 5, 64, "ln", torch.bfloat16, "silu"), (128, 2, 401, "ln", torch.float16, "silu")])
def test_chain_gradients(dev, many, C, num_layers, T, norm_kind, dtype, act):
    train.test_chain_gradients_against_fp32_torch_layers(dev, C, num_layers, T, norm_kind, dtype, act)


# two clouds each: the first token counts beyond the few-token limit, and either side of 32,768
@pytest.mark.parametrize("C,num_layers,T,norm_kind,dtype,act", [
    (128, 3, 6145, "ln", torch.bfloat16, "gelu"), (64, 6, 8193, "ln", torch.bfloat16, "silu"), (32, 6, 8193, "rms", torch.float16, "gelu"),
    (64, 3, 16384, "ln", torch.float16, "gelu"), (32, 3, 16385, "ln", torch.bfloat16, "silu")])
def test_chain_gradients_beyond_the_few_token_limit(dev, monkeypatch, C, num_layers, T, norm_kind, dtype, act):
    monkeypatch.setattr(fused, "_packed_few", _none_few)
    train.test_chain_gradients_against_fp32_torch_layers(dev, C, num_layers, T, norm_kind, dtype, act)


@pytest.mark.parametrize("C,T,xdt", [(64, 5000, torch.float32), (128, 3000, torch.bfloat16), (32, 1001, torch.float16)])
def test_pair_of_chains(dev, many, C, T, xdt):
    train.test_pair_of_chains_sums_its_input_gradients_in_the_second_launch(dev, C, T, xdt)


@pytest.mark.parametrize("C,num_layers,T", [(32, 6, 15), (64, 3, 17), (128, 3, 1), (128, 3, 4099)])
@pytest.mark.parametrize("kind,dtype,act", [("ln", torch.bfloat16, "gelu"), ("rms", torch.float16, "silu"), (None, torch.bfloat16, "gelu")])
def test_pair_of_alike_chains(dev, many, monkeypatch, C, num_layers, T, kind, dtype, act):
    real = fused._pair_info
    asked = []
    # the test under this one asserts that the few-token launch takes the pair: answer that question, and only that one
    monkeypatch.setattr(fused, "_pair_info", lambda *a: (asked.append(1), real(*a) or (() if len(asked) == 1 else None))[1])
    train.test_pair_of_chains_against_fp32_torch_layers(dev, C, num_layers, T, kind, dtype, act)
    assert len(asked) > 1


@pytest.mark.parametrize("C,H,M,N", [(64, 8, 64, 3000), (128, 8, 128, 2000), (32, 2, 32, 1000)])
def test_block_trains(dev, many, C, H, M, N):
    train.test_block_trains_through_the_fused_launches(dev, C, H, M, N)


@pytest.mark.parametrize("C,in_dim,out_dim,num_layers,T,norm_kind,dtype", [
    (128, 3, 128, 2, 3000, None, torch.bfloat16), (64, 64, 1, 2, 2500, "ln", torch.bfloat16), (32, 2, 4, 3, 777, None, torch.float16),
    (128, 128, 3, 3, 1100, "rms", torch.bfloat16)])
def test_narrow_end_stacks_train(dev, many, C, in_dim, out_dim, num_layers, T, norm_kind, dtype):
    train.test_narrow_end_stacks_train_through_the_fused_chain(dev, C, in_dim, out_dim, num_layers, T, norm_kind, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_16bit_parameters_residuals_and_order(dev, many, dtype):
    train.test_block_with_16bit_parameters_trains_fused(dev, dtype)
    train.test_separate_residual_and_no_residual(dev)
    train.test_detached_residual_over_the_rows_of_x(dev)
    train.test_backward_is_deterministic(dev)
