"""Block-sparse walks over 64 x 64 blocks (gemm_walk.hip) under the activation epilogues of LeanFFN: each compiled activation and one
chosen at run time, gated (two walks paired in one workgroup) and plain, tokens that end inside a 256-row tile, inside a wavefront's 64
rows and on their edge, a low-rank term of ragged length, lists longer than the registers hold.  All outputs and parameter gradients
against the fp32 CPU oracle at the 16-bit bars."""
import pytest
import torch

import lean_transformer_amd as lt
import test_gpu_sparse_paths  # noqa: F401  (registers the "scrambled" layout, which no rule about runs of blocks fits)
from test_gpu_ffn import _compare
from test_gpu_ffn_bf16_paths import _randomise_small_vectors

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def scrambled_ffn(hidden_blocks, inter_blocks, up_per_in, down_per_in, rank, act, gated):
    hidden, inter = 64 * hidden_blocks, 64 * inter_blocks
    up = lt.GeneralizedMatrix(hidden, 2 * inter if gated else inter, f"scrambled(per_in={up_per_in})", rank)
    down = lt.GeneralizedMatrix(inter, hidden, f"scrambled(per_in={down_per_in})", rank)
    ffn = lt.LeanFFN(hidden, inter, activation=lt.ACT2FN[act], gated=gated, layer_norm_eps=1e-5, i2h_proj=lt.GeneralizedLinear(up),
                     h2o_proj=lt.GeneralizedLinear(down))
    _randomise_small_vectors(ffn)
    return ffn


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["gelu_fused", "silu", "gelu", "mish"])
@pytest.mark.parametrize("gated,tokens", [(False, 257), (False, 300), (True, 257), (True, 300), (True, 320)])
def test_activations(dtype, act, gated, tokens):
    torch.manual_seed(tokens)
    ffn = scrambled_ffn(4, 8, 8 if gated else 4, 2, 24, act, gated).to(DEV).to(dtype)
    _compare(ffn, torch.randn(tokens, 256), torch.randn(tokens, 256), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("blocks,rank", [(66, 24),   # the second phase of the gated walk starts on a list of its own
                                         (132, 0)])  # both phases go on with a second list inside
def test_gated_walk_over_long_lists(dtype, blocks, rank):
    torch.manual_seed(blocks)
    ffn = scrambled_ffn(blocks, 2, 4, blocks, rank, "gelu_fused", True).to(DEV).to(dtype)
    _compare(ffn, torch.randn(70, 64 * blocks), torch.randn(70, 64 * blocks), dtype)
