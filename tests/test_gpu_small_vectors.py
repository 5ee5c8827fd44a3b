"""The small vectors of a block (LayerNorm parameters, biases) in the 16-bit compute dtype, which the library widens in one launch:
alignments and widths that are not multiples of anything, a mixture of dtypes and a strided one (converted one by one instead), and
the same figures from both."""
import pytest
import torch

import lean_transformer_amd as lt
from helpers import oracle_params, run_oracle
from conftest import assert_close
from test_gpu_ffn_bf16_paths import _randomise_small_vectors

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _step(ffn, x, dy):
    y = ffn(x)
    return [y, *torch.autograd.grad(y, [x, *ffn.parameters()], dy)]


@pytest.mark.parametrize("hidden,inter", [(8, 24), (100, 1025), (1032, 520)])
@pytest.mark.parametrize("post_ln", [False, True])
def test_widened_together_or_converted_one_by_one(hidden, inter, post_ln):
    torch.manual_seed(hidden)
    ffn = lt.LeanFFN(hidden, inter, gated=True, post_layer_norm=post_ln, layer_norm_eps=1e-5)
    _randomise_small_vectors(ffn)
    ffn = ffn.to(DEV).to(torch.bfloat16)
    x, dy = torch.randn(37, hidden), torch.randn(37, hidden)
    y_ref, dx_ref, _ = run_oracle(oracle_params(ffn), x, dy)
    xd, dyd = x.to(DEV).requires_grad_(True), dy.to(DEV)
    together = _step(ffn, xd, dyd)
    assert_close(together[0], y_ref, torch.bfloat16, "y")
    assert_close(together[1], dx_ref, torch.bfloat16, "dx")
    ffn.pre_layer_norm.weight.data = ffn.pre_layer_norm.weight.data.float()  # a mixture
    mixed = _step(ffn, xd, dyd)
    ffn.pre_layer_norm.weight.data = ffn.pre_layer_norm.weight.data.to(torch.bfloat16)
    ffn.i2h_proj.bias.data = torch.stack([ffn.i2h_proj.bias.data] * 2, 1)[:, 0]  # a strided one
    strided = _step(ffn, xd, dyd)
    for one, two, three in zip(together, mixed, strided):
        assert torch.equal(one, three) and torch.equal(one.float(), two.to(one.dtype).float())
