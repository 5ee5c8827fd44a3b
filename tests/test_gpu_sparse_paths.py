"""Block-sparse products over 64 x 64 blocks in 16 bits against float64 products with the dense matrix that the blocks make up: weight
gradients over runs of blocks with a shared list, their token reduction whole and split (more slices than whole ones, a short last one).

Bound: inputs are exact in float64, accumulation is fp32 (at most K + 16 additions, each off by 2^-23 of the magnitudes it adds) and
the result is rounded once to 16 bits (2^-9 of it in bfloat16, 2^-12 in float16, and its subnormal step)."""
import pytest
import torch

import lean_transformer_amd as lt

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.bfloat16: 2.0**-9, torch.float16: 2.0**-12}


def dense_weight(weight, backward_indices, out_features):
    """[out, in] float64 matrix of a native [in, A, 64] block-sparse weight (weight[ib * 64 + r, a] flat = block [64 out][64 in])"""
    in_features, per_in, block = weight.shape
    w4 = weight.detach().double().reshape(in_features // block, per_in, block, block)
    dense = torch.zeros(out_features, in_features, dtype=torch.float64, device=weight.device)
    for ib in range(in_features // block):
        for a in range(per_in):
            ob = int(backward_indices[ib, a])
            dense[ob * block:(ob + 1) * block, ib * block:(ib + 1) * block] = w4[ib, a]
    return dense


def blocks_of(dense, backward_indices, like):
    in_features, per_in, block = like.shape
    out = torch.empty(in_features // block, per_in, block, block, dtype=dense.dtype, device=dense.device)
    for ib in range(in_features // block):
        for a in range(per_in):
            ob = int(backward_indices[ib, a])
            out[ib, a] = dense[ob * block:(ob + 1) * block, ib * block:(ib + 1) * block]
    return out.reshape(like.shape)


def assert_bound(got, ref, magnitude, k, what):
    unit = UNIT[got.dtype]
    tiny = 2.0**-24 if got.dtype == torch.float16 else 0.0
    worst = (got.double() - ref).abs() - (k + 16) * 2.0**-23 * magnitude * (1 + unit) - unit * ref.abs() - tiny
    assert worst.max().item() <= 0.0, (what, worst.max().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("stretch", [True, False])
@pytest.mark.parametrize("in_f,out_f,tokens", [(512, 2048, 1000), (512, 2048, 2048), (512, 2048, 3333), (2048, 512, 2049), (1024, 4096, 9000)])
def test_weight_gradient(dtype, stretch, in_f, out_f, tokens):
    torch.manual_seed(tokens + in_f)
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(in_f, out_f, f"pixelfly(block_size=64, stretch={stretch})", 0), bias=False)
    layer = layer.to(DEV).to(dtype)
    x, dy = torch.randn(tokens, in_f, device=DEV).to(dtype), torch.randn(tokens, out_f, device=DEV).to(dtype)
    dw, = torch.autograd.grad(layer(x), layer.weight, dy)
    bwd = layer.matrix.backward_indices
    ref = blocks_of(dy.double().t() @ x.double(), bwd, dw)
    assert_bound(dw, ref, blocks_of(dy.double().abs().t() @ x.double().abs(), bwd, dw), tokens, "dw")
