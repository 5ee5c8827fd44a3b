"""16-bit products on 128 x 128 tiles (gemm_mid.hip): rows and columns around the tile and its 64-wide sub-tiles, reductions around the
8-element piece, the 64-k stage and the four stages in flight, one workgroup per CU and two (320 tiles), split reductions whose
last slice is short or empty.

Bound of test_gemm: fp32 accumulation of exact products, at most K + 16 additions each off by 2^-23 of the magnitudes it adds."""
import pytest
import torch

import lean_transformer_amd as lt
from conftest import assert_close
from helpers import oracle_params, run_oracle
from test_gpu_kernels import _gemm, _kernel_tags

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("a_kmajor,b_kmajor", [(True, True), (True, False), (False, False)])
@pytest.mark.parametrize("m,n,k", [(65, 8, 8), (127, 72, 64), (128, 128, 72), (129, 136, 192), (300, 264, 256), (192, 520, 264),
                                   (66, 64, 1000), (1000, 5000, 136)])
def test_gemm(dtype, a_kmajor, b_kmajor, m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = torch.randn(m, k, generator=g, device=DEV).to(dtype), torch.randn(n, k, generator=g, device=DEV).to(dtype)
    m8 = m if a_kmajor else -(-m // 8) * 8  # (an mn-major A has rows of a multiple of 8 elements)
    a = torch.cat([a, a[:m8 - m]])
    c, tags = _kernel_tags(lambda: _gemm(a if a_kmajor else a.t().contiguous(), b if b_kmajor else b.t().contiguous(), a_kmajor,
                                         b_kmajor, m8, n, k, torch.float32, 0))
    # (the tags are the bfloat16 library's; two mn-major operands go where the estimated time is the shorter)
    if dtype == torch.bfloat16 and a_kmajor:
        assert tags == {"gemm_mid_nt_store" if b_kmajor else "gemm_mid_nn_store"}, tags
    worst = (c.double() - a.double() @ b.double().t()).abs() - (k + 16) * 2.0**-23 * (a.double().abs() @ b.double().abs().t())
    assert worst.max().item() <= 0.0


@pytest.mark.parametrize("gated,dropout,post_ln", [(False, 0.0, False), (True, 0.0, True)])
@pytest.mark.parametrize("tokens,hidden,inter", [(65, 136, 2056), (130, 264, 8200), (513, 128, 1000)])
def test_split_reductions_of_a_training_step(gated, dropout, post_ln, tokens, hidden, inter):
    """the down-projection (its reduction is `inter`) and du (twice that when gated), through their summing passes"""
    torch.manual_seed(tokens)
    ffn = lt.LeanFFN(hidden, inter, gated=gated, post_layer_norm=post_ln, layer_norm_eps=1e-5).to(DEV).to(torch.bfloat16)
    x, dy = torch.randn(tokens, hidden), torch.randn(tokens, hidden)
    y_ref, dx_ref, g_ref = run_oracle(oracle_params(ffn), x, dy)
    xd = x.to(DEV).requires_grad_(True)

    def step():
        y = ffn(xd)
        return y, torch.autograd.grad(y, [xd, ffn.i2h_proj.weight, ffn.i2h_proj.bias, ffn.h2o_proj.weight], dy.to(DEV))

    (y, (dx, *grads)), tags = _kernel_tags(step)
    assert any(t.startswith("splitk_reduce") for t in tags), tags
    assert_close(y, y_ref, torch.bfloat16, "y")
    assert_close(dx, dx_ref, torch.bfloat16, "dx")
    for name, g, r in zip(("i2h.weight", "i2h.bias", "h2o.weight"), grads, g_ref[2:5]):
        assert_close(g, r, torch.bfloat16, name)


def test_long_reduction_of_many_tiles():
    """[1100, 4096] over 16384: 288 tiles of 128 x 128 leave the second workgroup of most CUs out; the down-projection and its input
    gradient run on 256 x 256 tiles in slices instead.  Against float32 products of the same 16-bit weights."""
    torch.manual_seed(0)
    tokens, hidden, inter = 1100, 4096, 16384
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN["linear"], gated=False, layer_norm_eps=1e-5).to(DEV).to(torch.bfloat16)
    x = torch.randn(tokens, hidden, device=DEV, requires_grad=True)
    dy = torch.randn(tokens, hidden, device=DEV)

    def step():
        y = ffn(x)
        return y.detach(), torch.autograd.grad(y, x, dy)[0]

    (y, dx), tags = _kernel_tags(step)
    assert {"gemm_bf16_nt_store", "splitk_reduce_out", "gemm_bf16_nn_store", "splitk_reduce"} <= tags, tags
    w1, b1, w2, b2 = (p.detach().float() for p in (ffn.i2h_proj.weight, ffn.i2h_proj.bias, ffn.h2o_proj.weight, ffn.h2o_proj.bias))
    u = torch.nn.functional.layer_norm(x, (hidden,), ffn.pre_layer_norm.weight.float(), ffn.pre_layer_norm.bias.float(), 1e-5)
    ref = (u @ w1.t() + b1) @ w2.t() + b2 + x
    ref_dx, = torch.autograd.grad(ref, x, dy)
    assert_close(y, ref.detach(), torch.bfloat16, "y")
    assert_close(dx, ref_dx, torch.bfloat16, "dx")
