"""Weight and low-rank gradients of one layer in one launch of 128 x 128 tiles: two and three of them, ragged reductions, one slice and many,
tiles of a few rows, and layers on either side of the 256 workgroups that share a launch."""
import pytest
import torch

from lean_transformer_amd import _native as nat
from lean_transformer_amd.blocksparse.linear import GeneralizedLinear, GeneralizedMatrix
from test_gpu_deferred_sums import test_gradients_summed_at_the_end as check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tokens,fan_in,fan_out,rank", [
    (65, 128, 128, 8),        # three products of a tile each, one slice
    (1000, 136, 264, 128),    # edges of tiles
    (4001, 640, 136, 136),    # a rank over one tile
    (2049, 768, 2304, 16),    # with the weight gradient where both fit 256 workgroups, the third alone
    (300, 2048, 2048, 24),    # 256 tiles of the weight gradient
    (300, 2176, 2048, 24),    # more: the low-rank pair alone
    (8200, 64, 64, 8),        # many slices
])
def test_gradients(tokens, fan_in, fan_out, rank):
    check(tokens, fan_in, fan_out, rank, True, "autocast")


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
