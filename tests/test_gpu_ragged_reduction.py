"""Reductions that do not end on a k-step of the tiled 16-bit kernels: the pieces past the end arrive as zeros from the buffer
unit's bounds check.  Reduction lengths around the 8-element piece, the 32-wide k-step and the 64-wide k-block; a second
k-segment (a low-rank term of any multiple of 8) behind a first that is padded to a whole block; a split reduction whose last
slice is ragged.  Bars: 1e-5 against a float64 product for fp32 results (sums of exactly representable products), the 16-bit
bars elsewhere."""
import pytest
import torch

import lean_transformer_amd as lt
from conftest import assert_close, rel_err
from helpers import oracle_params, run_oracle
from test_gpu_kernels import _gemm, _kernel_tags, _operands

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("a_kmajor,b_kmajor,tag", [(True, True, "gemm_bf16_nt_store"), (True, False, "gemm_bf16_nn_store"),
                                                   (False, False, "gemm_bf16_tn_store")])
@pytest.mark.parametrize("k", [8, 24, 32, 40, 56, 72, 96, 104, 128 + 8, 320 + 40, 1000])
def test_gemm_reduction_ends_inside_a_step(a_kmajor, b_kmajor, tag, k):
    m, n = 264, 264
    a, b, ref = _operands(m, n, k, a_kmajor, b_kmajor, torch.bfloat16, seed=k)
    c, tags = _kernel_tags(lambda: _gemm(a, b, a_kmajor, b_kmajor, m, n, k, torch.float32, 3))
    assert tag in tags, tags
    assert rel_err(c, ref) <= 1e-5


@pytest.mark.parametrize("features,rank", [((768, 2304), 16), ((200, 264), 8), ((1000, 520), 72)])
@pytest.mark.parametrize("tokens", [300, 4001])
def test_linear_with_a_ragged_low_rank_term(features, rank, tokens):
    """dense layer + adapter: the adapter's rank is the second k-segment; 4001 tokens split the weight gradients' reduction"""
    n_in, n_out = features
    torch.manual_seed(rank + tokens)
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(n_in, n_out), rank).to(DEV)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(std=0.05)
    layer = layer.to(torch.bfloat16)
    x = torch.randn(tokens, n_in, device=DEV).to(torch.bfloat16).requires_grad_(True)
    dy = torch.randn(tokens, n_out, device=DEV).to(torch.bfloat16)

    def step():
        y = layer(x)
        return y, torch.autograd.grad(y, [x, *layer.parameters()], dy)

    (y, grads), tags = _kernel_tags(step)
    assert "gemm_generic" not in tags, tags
    xr = x.detach().float().requires_grad_(True)
    ref = {name: p.detach().float().requires_grad_(True) for name, p in layer.named_parameters()}
    yr = xr @ ref["matrix.weight"].t() + ref["bias"] + (xr @ ref["adapter_first"].t()) @ ref["adapter_second"].t()
    refs = torch.autograd.grad(yr, [xr, *ref.values()], dy.float())
    assert_close(y, yr, torch.bfloat16, "y")
    for name, g, r in zip(["x", *ref], grads, refs):
        assert_close(g, r, torch.bfloat16, name)


@pytest.mark.parametrize("stretch", [True, False])
@pytest.mark.parametrize("rank,tokens", [(16, 300), (64, 1001)])
def test_sparse_ffn_with_ragged_tokens_and_rank(stretch, rank, tokens):
    """weight gradients over a token count no k-step divides (dense products over gathered blocks, skinny rank products), a
    rank below the k-step in the walks"""
    torch.manual_seed(rank + tokens)
    hidden, inter = 256, 1024
    layout = f"pixelfly(block_size=64, stretch={stretch})"
    up = lt.GeneralizedLinear(lt.GeneralizedMatrix(hidden, 2 * inter, layout, rank))
    down = lt.GeneralizedLinear(lt.GeneralizedMatrix(inter, hidden, layout, rank))
    ffn = lt.LeanFFN(hidden, inter, gated=True, layer_norm_eps=1e-5, i2h_proj=up, h2o_proj=down)
    with torch.no_grad():
        for p in (up.weight, down.weight, up.matrix.lowrank_first, up.matrix.lowrank_second, down.matrix.lowrank_first,
                  down.matrix.lowrank_second):
            p.normal_(std=0.05)
    ffn = ffn.to(DEV).to(torch.bfloat16)
    x, dy = torch.randn(tokens, hidden), torch.randn(tokens, hidden)
    y_ref, dx_ref, g_ref = run_oracle(oracle_params(ffn), x, dy)
    xd = x.to(DEV).requires_grad_(True)
    wanted = [xd, up.weight, up.matrix.lowrank_first, up.matrix.lowrank_second, down.weight, down.matrix.lowrank_first,
              down.matrix.lowrank_second]

    def step():
        y = ffn(xd)
        return y, torch.autograd.grad(y, wanted, dy.to(DEV))

    (y, grads), tags = _kernel_tags(step)
    assert not any("generic" in t for t in tags), tags
    assert_close(y, y_ref, torch.bfloat16, "y")
    # oracle parameter order: LN weight, LN bias, i2h weight, bias, first, second, h2o weight, bias, first, second
    refs = [dx_ref, g_ref[2], g_ref[4], g_ref[5], g_ref[6], g_ref[8], g_ref[9]]
    for name, g, r in zip(("dx", "dW1", "dL1a", "dL1b", "dW2", "dL2a", "dL2b"), grads, refs):
        assert_close(g, r, torch.bfloat16, name)
