"""Weight and low-rank gradients of one layer in one launch of 128 x 128 tiles: two and three of them, ragged reductions, one slice and many,
tiles of a few rows, and layers on either side of the 256 workgroups that share a launch."""
import pytest
import torch

from lean_transformer_amd import _native as nat
from lean_transformer_amd.blocksparse.linear import GeneralizedLinear, GeneralizedMatrix
from test_gpu_deferred_sums import check_whole_numbers, test_gradients_summed_at_the_end as check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# launches: of 128 x 128 tiles, for the weight gradient and the low-rank pair
@pytest.mark.parametrize("tokens,fan_in,fan_out,rank,launches", [
    (65, 128, 128, 8, 1),        # three products of a tile each, one slice
    (1000, 136, 264, 128, 1),    # edges of tiles
    (4001, 640, 136, 136, 1),    # a rank over one tile
    (2049, 768, 2304, 16, 1),    # 132 tiles, one slice
    (8200, 768, 2304, 16, 2),    # two slices: the weight gradient with the one that fits 256 workgroups beside it, the third alone
    (300, 2048, 2048, 24, 2),    # 256 tiles of the weight gradient: the low-rank pair alone
    (300, 2176, 2048, 24, 2),    # more
    (8200, 64, 64, 8, 1),        # many slices
])
def test_gradients(tokens, fan_in, fan_out, rank, launches):
    check(tokens, fan_in, fan_out, rank, True, "autocast")
    seen = check_whole_numbers(tokens, fan_in, fan_out, rank, True, "autocast")
    assert seen["gemm_mid_tn_store"] == launches, seen


def test_they_share_a_launch():
    torch.manual_seed(0)
    layer = GeneralizedLinear(GeneralizedMatrix(640, 384), adapter_dim=16, bias=False).to(DEV)
    x = torch.randn(4096, 640, device=DEV)
    with torch.autocast("cuda", torch.bfloat16):
        y = layer(x)
    lib = nat.lib(torch.bfloat16)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    torch.autograd.grad(y, list(layer.parameters()), torch.randn_like(y))
    lib.lt_profile_enable(0)
    launches = {tag: n for tag, n, *_ in nat.profile_read(lib)}
    assert launches["gemm_mid_tn_store"] == 1, launches
