"""Products of up to 64 rows (gemm_stream.hip): row counts around its 16-row tiles, column counts around its 16-column tiles and
on both sides of the lines between its workgroup shapes (up to 4096 weight rows, 32768 and more), reductions around its 16-byte
pieces and 128-byte blocks and shorter than its wavefronts.

Bound: fp32 accumulation of exact products, at most K + 16 additions each off by 2^-23 of the magnitudes it adds:
|c - ref| <= (K + 16) 2^-23 (|a| |b|^T)."""
import pytest
import torch

import lean_transformer_amd as lt
from helpers import dropout_mask, generator_position
from test_gpu_ffn import _compare
from test_gpu_ffn_bf16_paths import _randomise_small_vectors
from test_gpu_kernels import _gemm, _kernel_tags

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(4, 8), (20, 72), (264, 64), (260, 1000), (48, 8200), (4096, 40), (4100, 136), (32764, 136), (32768 + 8, 24)])
def test_gemm(dtype, m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = torch.randn(m, k, generator=g, device=DEV).to(dtype), torch.randn(n, k, generator=g, device=DEV).to(dtype)
    c, tags = _kernel_tags(lambda: _gemm(a, b, True, True, m, n, k, torch.float32, 0))
    assert dtype == torch.float16 or tags == {"gemm_stream"}, tags  # (the tags are the bfloat16 library's)
    worst = (c.double() - a.double() @ b.double().t()).abs() - (k + 16) * 2.0**-23 * (a.double().abs() @ b.double().abs().t())
    assert worst.max().item() <= 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 16, 21, 64])
@pytest.mark.parametrize("gated,act,dropout", [(True, "gelu_fused", 0.0), (False, "silu", 0.0), (True, "gelu", 0.1)])
@pytest.mark.parametrize("hidden,inter", [(104, 264), (256, 16384)])
def test_ffn(dtype, tokens, gated, act, dropout, hidden, inter):
    """every epilogue; 16384: the workgroup shape of many weight rows"""
    torch.manual_seed(tokens)
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN[act], gated=gated, dropout=dropout, layer_norm_eps=1e-5)
    _randomise_small_vectors(ffn)
    ffn = ffn.to(DEV).to(dtype)
    torch.cuda.manual_seed(5)
    mask = dropout_mask(tokens, hidden, dropout, *generator_position(DEV), torch.device(DEV)).cpu() if dropout else None
    _compare(ffn, torch.randn(tokens, hidden), torch.randn(tokens, hidden), dtype, mask=mask)


def test_rows_that_are_not_16_byte_aligned_take_another_kernel():
    a, b = torch.randn(3 * 40 + 1, device=DEV)[1:].view(3, 40), torch.randn(24, 40, device=DEV)
    c, tags = _kernel_tags(lambda: _gemm(a, b, True, True, 3, 24, 40, torch.float32, 0))
    assert tags == {"gemm_generic"} and torch.allclose(c, a @ b.t(), atol=1e-4)
