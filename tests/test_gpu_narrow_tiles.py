"""16-bit products on 256 x 192 tiles (launch_dma): whole ones, a last tile of 8 columns, rows and columns that stick out, reductions
around the k-step and the 64-k block, a second k-segment, workgroups that loop over tiles.

Bound of test_gemm: fp32 accumulation of exact products, at most K + 16 additions each off by 2^-23 of the magnitudes it adds."""
import pytest
import torch

import lean_transformer_amd as lt
from conftest import assert_close
from helpers import oracle_params, run_oracle
from lean_transformer_amd.ffn import philox_keep_mask
from test_gpu_kernels import _gemm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b_kmajor", [True, False])
@pytest.mark.parametrize("m,n,k", [(16384, 768, 64), (12300, 704, 200), (11000, 776, 72), (8200, 1160, 8), (8201, 1152, 1000),
                                   (16300, 2304, 328)])
def test_gemm(dtype, b_kmajor, m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = torch.randn(m, k, generator=g, device=DEV).to(dtype), torch.randn(n, k, generator=g, device=DEV).to(dtype)
    c = _gemm(a, b if b_kmajor else b.t().contiguous(), True, b_kmajor, m, n, k, torch.float32, 0)
    worst = (c.double() - a.double() @ b.double().t()).abs() - (k + 16) * 2.0**-23 * (a.double().abs() @ b.double().abs().t())
    assert worst.max().item() <= 0.0
    c16 = _gemm(a, b if b_kmajor else b.t().contiguous(), True, b_kmajor, m, n, k, dtype, 0)
    assert torch.equal(c16, c.to(dtype))


@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,hidden", [(12288, 768), (12301, 776)])
def test_down_projection_and_input_gradient(io, tokens, hidden):
    """residual epilogue, its dropout and the input gradient, whole tiles and ones that stick out; with dropout the elements that the
    mask drops are exactly the residual, and the rest agree with the unfused composition"""
    torch.manual_seed(tokens)
    ffn = lt.LeanFFN(hidden, 136, gated=True, layer_norm_eps=1e-5).to(DEV).to(torch.bfloat16)
    x, dy = torch.randn(tokens, hidden).to(io), torch.randn(tokens, hidden).to(io)
    y_ref, dx_ref, _ = run_oracle(oracle_params(ffn), x.float(), dy.float())
    xd = x.to(DEV).requires_grad_(True)
    y = ffn(xd)
    assert_close(y, y_ref, torch.bfloat16, "y")
    assert_close(torch.autograd.grad(y, xd, dy.to(DEV))[0], dx_ref, torch.bfloat16, "dx")
    if io == torch.float32:
        ffn = ffn.float()
        ffn.dropout = 0.5
        branch = []
        for custom in (True, False):
            ffn.ffn_custom_grad = custom
            torch.cuda.manual_seed(7)
            with torch.autocast("cuda", dtype=torch.bfloat16):
                branch.append((ffn(xd) - xd).detach())
        torch.cuda.manual_seed(7)
        keep = philox_keep_mask(tokens, hidden, 0.5, xd.device)
        assert (branch[0][keep == 0] == 0).all()
        assert_close(branch[0], branch[1].cpu(), torch.bfloat16, "branch under dropout")


def test_second_segment():
    """input gradient of a projection with a rank-16 adapter: g_hid L1 behind dy W, the first segment padded to a whole 64-k block"""
    torch.manual_seed(3)
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(776, 840), 16).to(DEV)
    torch.nn.init.normal_(layer.adapter_second, std=0.05)
    x, dy = torch.randn(12300, 776, device=DEV), torch.randn(12300, 840, device=DEV)
    w = (layer.weight + layer.adapter_second @ layer.adapter_first).double()
    xd = x.clone().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = layer(xd)
    assert_close(y, (x.double() @ w.t() + layer.bias.double()).float().cpu(), torch.bfloat16, "y")
    assert_close(torch.autograd.grad(y, xd, dy.to(y.dtype))[0], (dy.double() @ w).float().cpu(), torch.bfloat16, "dx")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(256, 136, 32), (264, 776, 33), (1600, 1608, 333), (8, 328, 7), (6400, 1600, 129)])
def test_weight_gradient(dtype, m, n, k):
    """both operands mn-major; the bound of test_gemm"""
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = torch.randn(k, m, generator=g, device=DEV).to(dtype), torch.randn(k, n, generator=g, device=DEV).to(dtype)
    c = _gemm(a, b, False, False, m, n, k, torch.float32, 3)
    worst = (c.double() - a.double().t() @ b.double()).abs() - (k + 16) * 2.0**-23 * (a.double().abs().t() @ b.double().abs())
    assert worst.max().item() <= 0.0
