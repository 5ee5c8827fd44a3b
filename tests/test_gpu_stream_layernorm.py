"""Blocks of a few rows, whose LayerNorm is part of the up-projection: against the oracle, gradients (which read the statistics it leaves)
among them, at the edges of rows, widths and the three workgroup shapes, and rows alone against the same rows in larger batches."""
import pytest
import torch

import lean_transformer_amd as lt
from helpers import oracle_params, run_oracle
from conftest import assert_close
from lean_transformer_amd import _native as nat
from test_gpu_ffn_bf16_paths import _randomise_small_vectors

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ffn(hidden, inter, gated, dtype, **kw):
    torch.manual_seed(hidden + inter)
    ffn = lt.LeanFFN(hidden, inter, gated=gated, layer_norm_eps=1e-5, **kw)
    _randomise_small_vectors(ffn)
    return ffn.to(DEV).to(dtype)


# (inter decides the workgroup shape: up to 4096 plain rows of weights, at least 32768, between)
@pytest.mark.parametrize("tokens", [1, 2, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("hidden,inter,gated", [(8, 16, True), (104, 1000, False), (520, 2056, True), (1032, 64, False), (4096, 256, True), (1024, 512, True),
                                                (64, 32768, False), (72, 16400, True)])
@pytest.mark.parametrize("dtype,stream", [(torch.float32, "same"), (torch.bfloat16, "same"), (torch.bfloat16, "fp32"), (torch.float16, "same"),
                                          (torch.float16, "fp32")])
def test_few_rows_against_the_oracle(tokens, hidden, inter, gated, dtype, stream):
    ffn = _ffn(hidden, inter, gated, dtype)
    io = dtype if stream == "same" else torch.float32
    x, dy = (3 * torch.randn(tokens, hidden) + 1).to(io).float(), torch.randn(tokens, hidden).to(io).float()
    y_ref, dx_ref, g_ref = run_oracle(oracle_params(ffn), x, dy)
    xd = x.to(DEV).to(io).requires_grad_(True)
    lib = nat.lib(dtype)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    y = ffn(xd)
    lib.lt_profile_enable(0)
    size = torch.empty(0, dtype=dtype).element_size()
    inside = tokens <= (8 if size == 2 else 4) and tokens * hidden * size <= 32768  # rows, and what LDS keeps of them
    assert {e[0] for e in nat.profile_read(lib)} == ({"gemm_stream"} if inside else {"gemm_stream", "layernorm_fwd"})
    dx, dw1 = torch.autograd.grad(y, [xd, ffn.i2h_proj.weight], dy.to(DEV).to(io))
    assert_close(y, y_ref, dtype, "y")
    assert_close(dx, dx_ref, dtype, "dx")
    assert_close(dw1, g_ref[2], dtype, "dW1")


@pytest.mark.parametrize("case", ["autocast", "mixed vectors", "odd address", "wide", "ragged", "post_ln", "rows"])
def test_neighbours_of_the_rule(case):
    """what the rule leaves out or takes with vectors in fp32"""
    hidden = {"wide": 4104, "ragged": 100}.get(case, 256)
    ffn = _ffn(hidden, 512, True, torch.float32 if case == "autocast" else torch.bfloat16, post_layer_norm=case == "post_ln")
    if case == "mixed vectors":
        ffn.pre_layer_norm.weight.data = ffn.pre_layer_norm.weight.data.float()
    if case == "odd address":
        flat = torch.empty(hidden + 1, dtype=torch.bfloat16, device=DEV)
        flat[1:].copy_(ffn.pre_layer_norm.bias.data)
        ffn.pre_layer_norm.bias.data = flat[1:]
    tokens = 9 if case == "rows" else 3
    x, dy = torch.randn(tokens, hidden), torch.randn(tokens, hidden)
    y_ref, dx_ref, _ = run_oracle(oracle_params(ffn), x, dy)
    xd = x.to(DEV).requires_grad_(True)
    with torch.autocast("cuda", torch.bfloat16, enabled=case == "autocast"):
        y = ffn(xd)
    dx, = torch.autograd.grad(y, xd, dy.to(DEV))
    assert_close(y, y_ref, torch.bfloat16, "y")
    assert_close(dx, dx_ref, torch.bfloat16, "dx")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_with_infinities(dtype):
    """a row that overflows leaves the others alone, and comes out as in the general path"""
    ffn = _ffn(64, 128, True, dtype)
    x = torch.randn(5, 64).to(dtype)
    x[2, 7] = float("inf")
    x[3, 1] = float("nan")
    with torch.no_grad():
        few, many = ffn(x.to(DEV)), ffn(torch.cat([x, torch.randn(20, 64).to(dtype)]).to(DEV))[:5]
    assert torch.equal(few.isnan(), many.isnan()) and few[2:4].isnan().all() and not few[[0, 1, 4]].isnan().any()
    keep = [0, 1, 4]
    assert_close(few[keep], many[keep].float().cpu(), dtype, "y")


@pytest.mark.parametrize("hidden,inter,gated", [(104, 1000, False), (520, 2056, True), (64, 32768, False)])
@pytest.mark.parametrize("dtype,most", [(torch.float32, 4), (torch.bfloat16, 8), (torch.float16, 8)])
def test_rows_alone_and_in_larger_batches(hidden, inter, gated, dtype, most):
    """the same bits for a row in every batch that is taken; above, its LayerNorm is summed in another order (one wavefront a row)"""
    ffn = _ffn(hidden, inter, gated, dtype)
    x = (3 * torch.randn(24, hidden) + 1).to(dtype).to(DEV)
    with torch.no_grad():
        rows = torch.cat([ffn(x[i:i + 1]) for i in range(most)])
        for tokens in (2, 3, most):
            assert torch.equal(ffn(x[:tokens]), rows[:tokens]), tokens
        for tokens in (most + 1, 24):
            assert_close(ffn(x[:tokens])[:most], rows.cpu(), dtype, "y")
