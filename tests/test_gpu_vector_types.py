"""LayerNorm parameters read in 16 bits and gradients of the small vectors written in 16 bits: the same figures as from vectors at odd
addresses, which are widened first, and the fp32 gradients rounded once."""
import pytest
import torch

import lean_transformer_amd as lt
from lean_transformer_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _at_odd_address(param):
    flat = torch.empty(param.numel() + 1, dtype=param.dtype, device=DEV)
    flat[1:].copy_(param.detach().flatten())
    return torch.nn.Parameter(flat[1:].view(param.shape))


# 8200: wider than the register-resident rows; 1030, 102: no 16-byte pieces; 4100: two backward kernels; 2056: two wavefronts a row
@pytest.mark.parametrize("tokens,hidden", [(1, 8), (5, 102), (70, 1030), (33, 2056), (9, 4100), (3, 8200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("stream", ["fp32", "same"])
@pytest.mark.parametrize("post_ln", [False, True])
def test_vectors_as_they_are(tokens, hidden, dtype, stream, post_ln):
    torch.manual_seed(hidden)
    ffn = lt.LeanFFN(hidden, 24, post_layer_norm=post_ln, gated=True, layer_norm_eps=1e-5).to(DEV)
    with torch.no_grad():
        for name, p in ffn.named_parameters():
            if p.dim() == 1:
                p.add_(torch.randn_like(p) * 0.5)
    ffn = ffn.to(dtype)
    io = torch.float32 if stream == "fp32" else dtype
    x = torch.randn(tokens, hidden, device=DEV).to(io).requires_grad_(True)
    dy = torch.randn(tokens, hidden, device=DEV).to(io)

    def step():
        y = ffn(x)
        return [y.detach(), *torch.autograd.grad(y, [x, *ffn.parameters()], dy)]

    plain = step()
    for module in ffn.modules():
        for name in ("weight", "bias"):
            p = getattr(module, name, None)
            if p is not None and p.dim() == 1:
                setattr(module, name, _at_odd_address(p))
                assert getattr(module, name).data_ptr() % 4 == 2
    shifted = step()
    for a, b, name in zip(plain, shifted, ["y", "x", *(n for n, _ in ffn.named_parameters())]):
        assert a.dtype == b.dtype and torch.equal(a, b), (name, (a.float() - b.float()).abs().max().item())


@pytest.mark.parametrize("tokens,hidden,inter", [(1, 8, 16), (66, 132, 264), (700, 768, 3072)])
def test_gradients_of_vectors_are_the_fp32_ones_rounded(tokens, hidden, inter):
    torch.manual_seed(tokens)
    ffn = lt.LeanFFN(hidden, inter, gated=True, post_layer_norm=True, layer_norm_eps=1e-5).to(DEV).to(torch.bfloat16)
    x = torch.randn(tokens, hidden, device=DEV, requires_grad=True)
    dy = torch.randn(tokens, hidden, device=DEV)
    vectors = [ffn.pre_layer_norm.weight, ffn.pre_layer_norm.bias, ffn.post_layer_norm.weight, ffn.post_layer_norm.bias,
               ffn.i2h_proj.bias, ffn.h2o_proj.bias]
    y = ffn(x)
    half = torch.autograd.grad(y, vectors, dy)
    lib, seen = nat.lib(torch.bfloat16), {}
    original = lib.lt_ffn_backward_typed

    def in_fp32(desc, px, pdy, saved, grads, grad_dtype, vector_dtype, *rest):
        """the same call with the vectors' gradients in fp32, into a buffer of its own"""
        assert vector_dtype == nat.LT_BF16
        for name, n in (("ln_weight", hidden), ("ln_bias", hidden), ("post_ln_weight", hidden), ("post_ln_bias", hidden)):
            seen[name] = torch.empty(n, device=DEV)
            setattr(grads, name, seen[name].data_ptr())
        for name, n in (("i2h", 2 * inter), ("h2o", hidden)):
            seen[name] = torch.empty(n, device=DEV)
            getattr(grads, name).bias = seen[name].data_ptr()
        return original(desc, px, pdy, saved, grads, grad_dtype, nat.LT_F32, *rest)

    y = ffn(x)
    try:
        lib.lt_ffn_backward_typed = in_fp32
        torch.autograd.grad(y, vectors, dy)
    finally:
        lib.lt_ffn_backward_typed = original
    for g, name in zip(half, ("ln_weight", "ln_bias", "post_ln_weight", "post_ln_bias", "i2h", "h2o")):
        assert g.dtype == torch.bfloat16 and torch.equal(g, seen[name].bfloat16()), name
