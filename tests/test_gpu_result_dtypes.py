"""fp32 parameters under autocast: input and weight gradients leave the kernels in fp32.  The same products in the same order as for a
module in the 16-bit type itself, only stored before the last rounding: rounded, they are that module's gradients bit for bit."""
import copy

import pytest
import torch

import lean_transformer_amd as lt

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
STRETCHED, TILED = "pixelfly(block_size=64, stretch=True)", "pixelfly(block_size=64)"


def _both(module, x, dtype, io_follows):
    """gradients (input's first) of the fp32 module under autocast and of its copy in `dtype`; parameters fit both types"""
    with torch.no_grad():
        for p in module.parameters():
            p.normal_(std=0.05)
            p.copy_(p.to(dtype))
    low = copy.deepcopy(module).to(dtype)
    results = []
    for m, autocast, leaf in ((module, True, x), (low, False, x.to(dtype) if io_follows else x)):
        leaf = leaf.detach().clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=dtype, enabled=autocast):
            y = m(leaf)
        torch.manual_seed(5)
        dy = torch.randn(y.shape, device=DEV).to(y.dtype)
        results.append((y.detach(), torch.autograd.grad(y, [leaf, *m.parameters()], dy)))
    return results


def _compare(results, dtype, names):
    (y, wide), (y_low, low) = results
    assert torch.equal(y.to(dtype), y_low.to(dtype))
    unrounded = 0
    for name, a, b in zip(names, wide, low):
        assert a.dtype == torch.float32, name
        assert torch.equal(a.to(dtype), b.to(dtype)), name
        unrounded += not torch.equal(a, a.to(dtype).float())
    assert unrounded >= 2  # (the types differ for a reason)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,in_f,out_f,rank,layout", [
    (5, 64, 96, 0, None), (40, 512, 256, 8, None), (33, 72, 200, 16, None),  # few rows; any shape
    (700, 768, 2304, 16, None), (3333, 1600, 1608, 0, None),                  # 128 x 128 tiles; sizes off the grid
    (4096, 2048, 2048, 64, None), (8192, 2048, 8192, 128, None),              # 256 x 256 tiles, split and whole
    (300, 256, 1024, 0, STRETCHED), (2049, 1024, 256, 64, STRETCHED), (2049, 512, 2048, 16, TILED), (33, 256, 256, 0, STRETCHED)])
def test_linear(dtype, tokens, in_f, out_f, rank, layout):
    torch.manual_seed(tokens)
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(in_f, out_f, layout, rank)).to(DEV)
    names = ["input", *(n for n, _ in layer.named_parameters())]
    _compare(_both(layer, torch.randn(tokens, in_f, device=DEV).to(dtype).float(), dtype, True), dtype, names)


@pytest.mark.parametrize("tokens,hidden,inter,layout,rank", [(37, 96, 160, None, 0), (3000, 768, 3072, None, 0), (1000, 512, 2048, TILED, 64)])
def test_ffn(tokens, hidden, inter, layout, rank):
    torch.manual_seed(tokens)
    projections = {}
    if layout:
        projections = dict(i2h_proj=lt.GeneralizedLinear(lt.GeneralizedMatrix(hidden, 2 * inter, layout, rank)),
                           h2o_proj=lt.GeneralizedLinear(lt.GeneralizedMatrix(inter, hidden, layout, rank)))
    layer = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN["gelu_fused"], gated=True, **projections).to(DEV)
    names = ["input", *(n for n, _ in layer.named_parameters())]
    _compare(_both(layer, torch.randn(tokens, hidden, device=DEV), torch.bfloat16, False), torch.bfloat16, names)


def test_only_the_compute_type_and_fp32_are_taken():
    from lean_transformer_amd import _native as nat
    from lean_transformer_amd.blocksparse.linear import linear_desc
    w, x = torch.zeros(64, 64, device=DEV, dtype=torch.float32), torch.zeros(8, 64, device=DEV)
    desc, grads, lib = linear_desc(w, None, None, None, None, None), nat.LtLinearGrads(), nat.lib()
    ws = nat.workspace(lib.lt_linear_backward_workspace_bytes(desc, 8, nat.LT_F32), w.device)
    for dx_dtype, grad_dtype in ((nat.LT_BF16, nat.LT_F32), (nat.LT_F32, nat.LT_BF16)):
        assert lib.lt_linear_backward_to(desc, 8, nat.LT_F32, nat.ptr(x), nat.ptr(x), None, dx_dtype, nat.ptr(x), grads, grad_dtype,
                                         nat.ptr(ws), ws.numel(), nat.current_stream(w.device)) != 0
