"""Products on more 128 x 128 tiles than run at once: forward, input gradient and the bias gradient that the latter's epilogue
sums, at ragged rows and columns, and the whole rounds of 256 x 256 tiles that stay with the other kernel."""
import pytest
import torch

import lean_transformer_amd as lt
from conftest import assert_close
from helpers import dropout_mask, generator_position, oracle_params, run_oracle
from lean_transformer_amd import _native as nat
from test_gpu_ffn_bf16_paths import _randomise_small_vectors

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,hidden,inter,gated,act,kernel", [
    (5500, 512, 2048, False, "silu", "mid"),       # 176 tiles of 256 x 256
    (4231, 264, 3080, False, "gelu", "mid"),       # columns off the 64-wide sub-tiles, the last row tile of seven rows
    (1601, 392, 2568, True, "gelu_fused", "mid"),  # gated pairs off the tile
    (8192, 2048, 2048, False, "silu", "bf16"),     # 256 tiles: one whole round
])
def test_activation_epilogues(dtype, tokens, hidden, inter, gated, act, kernel):
    torch.manual_seed(tokens)
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN[act], gated=gated, layer_norm_eps=1e-5)
    _randomise_small_vectors(ffn)
    ffn = ffn.to(DEV).to(dtype)
    x, dy = torch.randn(tokens, hidden), torch.randn(tokens, hidden)
    y_ref, dx_ref, g_ref = run_oracle(oracle_params(ffn), x, dy)
    xd = x.to(DEV).requires_grad_(True)
    lib = nat.lib(dtype)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    y = ffn(xd)
    dx, dw1, db1, dw2 = torch.autograd.grad(y, [xd, ffn.i2h_proj.weight, ffn.i2h_proj.bias, ffn.h2o_proj.weight], dy.to(DEV))
    lib.lt_profile_enable(0)
    tags = {e[0] for e in nat.profile_read(lib)}
    assert f"gemm_{kernel}_nt_act_fwd" in tags and (gated or f"gemm_{kernel}_nn_act_bwd" in tags), tags
    for name, got, ref in (("y", y, y_ref), ("dx", dx, dx_ref), ("dW1", dw1, g_ref[2]), ("db1", db1, g_ref[3]), ("dW2", dw2, g_ref[4])):
        assert_close(got, ref, dtype, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dropout", [0.0, 0.2])
def test_unfused_products_and_down_projection(dtype, dropout):
    """272 tiles of 256 x 256 for 256 compute units: down-projection and du on 1139 of 128 x 128, ragged in rows and columns"""
    tokens, hidden, inter = 8449, 2040, 776
    torch.manual_seed(5)
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN["silu"], layer_norm_eps=1e-5, dropout=dropout)
    _randomise_small_vectors(ffn)
    ffn = ffn.to(DEV).to(dtype)
    x, dy = torch.randn(tokens, hidden), torch.randn(tokens, hidden)
    mask = None
    if dropout:
        mask = dropout_mask(tokens, hidden, dropout, *generator_position(DEV), torch.device(DEV)).cpu()
    y_ref, dx_ref, g_ref = run_oracle(oracle_params(ffn), x, dy, mask)
    xd = x.to(DEV).requires_grad_(True)
    lib = nat.lib(dtype)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    y = ffn(xd)
    dx, dw2 = torch.autograd.grad(y, [xd, ffn.h2o_proj.weight], dy.to(DEV))
    lib.lt_profile_enable(0)
    tags = {e[0] for e in nat.profile_read(lib)}
    assert {"gemm_mid_nt_out", "gemm_mid_nn_store"} <= tags, tags
    for name, got, ref in (("y", y, y_ref), ("dx", dx, dx_ref), ("dW2", dw2, g_ref[4])):
        assert_close(got, ref, dtype, name)


@pytest.mark.parametrize("tokens,hidden,inter,forward,backward", [
    (1100, 2048, 8192, "mid", "mid"),    # 160 tiles of 256 x 256
    (563, 2056, 14776, "bf16", "mid"),   # a longer reduction
    (889, 3584, 10048, "bf16", "mid"),
    (2203, 4096, 5176, "bf16", "bf16"),  # 189 tiles, the longest
    (2203, 4096, 8200, "mid", "mid"),    # 297: more than one round
])
def test_long_reductions_that_leave_compute_units_idle(tokens, hidden, inter, forward, backward):
    """which kernel takes the two activation epilogues (what it computes is the other tests' matter)"""
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN["silu"]).to(DEV).to(torch.bfloat16)
    x = torch.randn(tokens, hidden, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    lib = nat.lib(torch.bfloat16)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    torch.autograd.grad(ffn(x), x, torch.randn_like(x))
    lib.lt_profile_enable(0)
    tags = {e[0] for e in nat.profile_read(lib)}
    assert {f"gemm_{forward}_nt_act_fwd", f"gemm_{backward}_nn_act_bwd"} <= tags, tags


@pytest.mark.parametrize("tokens,hidden,inter,out,input_gradient", [
    (9528, 1600, 792, "mid", "mid"),    # 266 tiles of 256 x 256: a second round of ten
    (8541, 2376, 1208, "mid", "bf16"),  # a third of a second round
    (16384, 2048, 1024, "bf16", "bf16"),  # two whole rounds
])
def test_unfused_products_by_rounds(tokens, hidden, inter, out, input_gradient):
    """which kernel takes the down-projection and the up-projection's input gradient"""
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN["silu"]).to(DEV).to(torch.bfloat16)
    x = torch.randn(tokens, hidden, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    lib = nat.lib(torch.bfloat16)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    torch.autograd.grad(ffn(x), x, torch.randn_like(x))
    lib.lt_profile_enable(0)
    tags = {e[0] for e in nat.profile_read(lib)}
    assert {f"gemm_{out}_nt_out", f"gemm_{input_gradient}_nn_store"} <= tags, tags
