"""Activation epilogues of the copy-based 16-bit kernels where tiles stick out: the last rows (300 = 256 + 44, 8236 = 32 x 256 + 44), a
column tile of 8 (264, 520, 1032 = a multiple of 256 + 8) and the gated pairing's half-width tile (520 and 1032, of 128 + 8), on
128 x 128 tiles (300 rows) and 256 x 256 ones (8236), for the activations with a kernel of their
own (the tanh GELU, SiLU, the exact GELU) and one that shares the run-time choice (mish).  Bars: the 16-bit ones."""
import pytest
import torch

import lean_transformer_amd as lt
from lean_transformer_amd.utils import ACT2FN
from test_gpu_ffn import _compare
from test_gpu_ffn_bf16_paths import _randomise_small_vectors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("act", ["gelu_fused", "silu", "gelu", "mish"])
@pytest.mark.parametrize("tokens,hidden,inter", [(300, 264, 520), (300, 256, 512), (8236, 1032, 1032)])
def test_activation_epilogues_at_the_edges(act, gated, tokens, hidden, inter):
    torch.manual_seed(31)
    ffn = lt.LeanFFN(hidden, inter, activation=ACT2FN[act], gated=gated, layer_norm_eps=1e-5)
    _randomise_small_vectors(ffn)
    ffn = ffn.to("cuda:0").to(torch.bfloat16)
    _compare(ffn, torch.randn(tokens, hidden), torch.randn(tokens, hidden), torch.bfloat16)
