"""Block-sparse products over 64 x 64 blocks in 16 bits against float64 products with the dense matrix that the blocks make up: weight
gradients over runs of blocks with a shared list, their token reduction whole and split (more slices than whole ones, a short last one).

Bound: inputs are exact in float64, accumulation is fp32 (at most K + 16 additions, each off by 2^-23 of the magnitudes it adds) and
the result is rounded once to 16 bits (half a unit in the last place: 2^-8 of it with the 8 significant bits of bfloat16,
2^-11 with the 11 of float16, and half its subnormal step, 2^-25)."""
import pytest
import torch

import lean_transformer_amd as lt
from test_gpu_ffn import _compare
from test_gpu_kernels import _kernel_tags

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def dense_weight(weight, backward_indices, out_features):
    """[out, in] float64 matrix of a native [in, A, 64] block-sparse weight (weight[ib * 64 + r, a] flat = block [64 out][64 in])"""
    in_features, per_in, block = weight.shape
    w4 = weight.detach().double().reshape(in_features // block, per_in, block, block)
    dense = torch.zeros(out_features, in_features, dtype=torch.float64, device=weight.device)
    for ib in range(in_features // block):
        for a in range(per_in):
            ob = int(backward_indices[ib, a])
            dense[ob * block:(ob + 1) * block, ib * block:(ib + 1) * block] = w4[ib, a]
    return dense


def blocks_of(dense, backward_indices, like):
    in_features, per_in, block = like.shape
    out = torch.empty(in_features // block, per_in, block, block, dtype=dense.dtype, device=dense.device)
    for ib in range(in_features // block):
        for a in range(per_in):
            ob = int(backward_indices[ib, a])
            out[ib, a] = dense[ob * block:(ob + 1) * block, ib * block:(ib + 1) * block]
    return out.reshape(like.shape)


def assert_bound(got, ref, magnitude, k, what):
    unit = UNIT[got.dtype]
    tiny = 2.0**-24 if got.dtype == torch.float16 else 0.0
    worst = (got.double() - ref).abs() - (k + 16) * 2.0**-23 * magnitude * (1 + unit) - unit * ref.abs() - tiny
    assert worst.max().item() <= 0.0, (what, worst.max().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("stretch", [True, False])
@pytest.mark.parametrize("in_f,out_f,tokens", [(512, 2048, 1000), (512, 2048, 2048), (512, 2048, 3333), (2048, 512, 2049), (1024, 4096, 9000)])
def test_weight_gradient(dtype, stretch, in_f, out_f, tokens):
    torch.manual_seed(tokens + in_f)
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(in_f, out_f, f"pixelfly(block_size=64, stretch={stretch})", 0), bias=False)
    layer = layer.to(DEV).to(dtype)
    x, dy = torch.randn(tokens, in_f, device=DEV).to(dtype), torch.randn(tokens, out_f, device=DEV).to(dtype)
    dw, = torch.autograd.grad(layer(x), layer.weight, dy)
    bwd = layer.matrix.backward_indices
    ref = blocks_of(dy.double().t() @ x.double(), bwd, dw)
    assert_bound(dw, ref, blocks_of(dy.double().abs().t() @ x.double().abs(), bwd, dw), tokens, "dw")


@lt.blocksparse.layout.register_blocksparse_layout("scrambled")
def scrambled_layout(out_features, in_features, per_in):
    """a balanced layout that no rule about runs fits: `per_in` output blocks to each input block, in scrambled order"""
    in_blocks, out_blocks = in_features // 64, out_features // 64
    shift = torch.randperm(out_blocks, generator=torch.Generator().manual_seed(per_in))
    layout = torch.zeros(out_blocks, in_blocks, dtype=torch.bool)
    for ib in range(in_blocks):
        layout[shift[torch.arange(ib * per_in, (ib + 1) * per_in) % out_blocks], ib] = True
    return layout


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("in_blocks,out_blocks,per_in,rank,tokens", [
    (4, 4, 1, 0, 1),          # one step
    (4, 8, 6, 8, 255),        # a short low-rank step behind an odd list
    (8, 4, 2, 64, 257),       # rows that stick out
    (16, 16, 5, 72, 513),     # low-rank term of more than one step, the last one short
    (2, 66, 66, 16, 300),     # a list longer than one register
    (132, 66, 33, 0, 4200),   # two workgroups per CU
    (2, 132, 132, 24, 70),    # lists too long for the registers
    (132, 2, 2, 24, 70)])
def test_forward_and_input_gradient(dtype, in_blocks, out_blocks, per_in, rank, tokens):
    """walks over lists of 1 to 132 blocks, in both pipeline depths, with a low-rank term of ragged length.  The term's intermediate is
    rounded to 16 bits: its magnitude times the unit, through the second factor, joins the bound."""
    torch.manual_seed(tokens + rank)
    in_f, out_f = 64 * in_blocks, 64 * out_blocks
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(in_f, out_f, f"scrambled(per_in={per_in})", rank), bias=False).to(DEV).to(dtype)
    x, dy = torch.randn(tokens, in_f, device=DEV).to(dtype).requires_grad_(True), torch.randn(tokens, out_f, device=DEV).to(dtype)
    y = layer(x)
    dx, = torch.autograd.grad(y, x, dy)
    w = dense_weight(layer.weight, layer.matrix.backward_indices, out_f)
    l1, l2 = (t.detach().double() for t in (layer.matrix.lowrank_first, layer.matrix.lowrank_second)) if rank else (w[:0], w[:, :0])
    k = max(in_f, out_f) + rank
    for got, v, m, first, second in ((y, x.detach().double(), w.t(), l1.t(), l2.t()), (dx, dy.double(), w, l2, l1)):
        hid = v @ first
        ref, magnitude = v @ m + hid @ second, v.abs() @ m.abs() + hid.abs() @ second.abs()
        slack = 2 * UNIT[dtype] * hid.abs() @ second.abs() + (k + 16) * 2.0**-22 * (v.abs() @ first.abs()) @ second.abs()
        unit, tiny = UNIT[dtype], 2.0**-24 if dtype == torch.float16 else 0.0
        worst = (got.double() - ref).abs() - ((k + 16) * 2.0**-23 * magnitude + slack) * (1 + unit) - unit * ref.abs() - tiny
        assert worst.max().item() <= 0.0, worst.max().item()


@pytest.mark.parametrize("tokens", [10240, 10248])
def test_gated_up_projection_on_either_side_of_the_rule(tokens):
    """a stretched butterfly of hidden 1024: up to 160 MiB of pre-activation the paired walk, above that 256 x 256 tiles and an activation
    pass.  The normalised input, the pre-activation, the hidden activation and the weights' products of it are each off by at
    most a unit (2^-8) relative to their own 2-norm."""
    import oracle.ffn as offn
    torch.manual_seed(3)
    layout = "pixelfly(block_size=64, stretch=True)"
    up, down = (lt.GeneralizedLinear(lt.GeneralizedMatrix(i, o, layout)) for i, o in ((1024, 8192), (4096, 1024)))
    layer = lt.LeanFFN(1024, 4096, activation=lt.ACT2FN["gelu_fused"], gated=True, i2h_proj=up, h2o_proj=down)
    layer = layer.to(DEV).to(torch.bfloat16).eval()
    x = torch.randn(tokens, 1024, device=DEV)
    with torch.no_grad():
        y = layer(x) - x
        rows = torch.cat([torch.arange(64), torch.arange(tokens - 64, tokens)]).to(DEV)
        u = torch.nn.functional.layer_norm(x[rows].double(), (1024,))
        pre = u @ dense_weight(up.weight, up.matrix.backward_indices, 8192).t()
        hid = offn.apply_activation(pre, "gelu_fused", True)
        ref = hid @ dense_weight(down.weight, down.matrix.backward_indices, 1024).t()
    assert (y[rows].double() - ref).norm() <= 4 * 2.0**-8 * ref.norm()


@pytest.mark.parametrize("tokens,two_passes", [(20480, False), (20488, True)])
def test_gated_up_projection_on_either_side_of_the_rule_with_gradients(tokens, two_passes):
    """a stretched butterfly of hidden 512 with a low-rank term (of whole 64s, or the walk takes it in any case), 160 MiB of
    pre-activation and a little more: outputs and all gradients
    against the fp32 oracle at the bf16 bars, and which way the launch went"""
    torch.manual_seed(tokens)
    layout = "pixelfly(block_size=64, stretch=True)"
    up, down = (lt.GeneralizedLinear(lt.GeneralizedMatrix(i, o, layout, 64)) for i, o in ((512, 4096), (2048, 512)))
    layer = lt.LeanFFN(512, 2048, gated=True, layer_norm_eps=1e-5, i2h_proj=up, h2o_proj=down).to(DEV).to(torch.bfloat16)
    x, dy = torch.randn(tokens, 512), torch.randn(tokens, 512)
    _, tags = _kernel_tags(lambda: layer(x.to(DEV)))
    assert ("activation_fwd" in tags) == two_passes, tags
    _compare(layer, x, dy, torch.bfloat16, oracle_device=DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_equal_rows_in_different_token_tiles(dtype):
    """a walk starts its list at another entry in each 256-token tile, so that equal rows are summed in different orders and may differ
    in their last bits: by no more than the two roundings and the two fp32 sums' bounds"""
    torch.manual_seed(1)
    layer = lt.GeneralizedLinear(lt.GeneralizedMatrix(1024, 1024, "scrambled(per_in=12)", 0), bias=False).to(DEV).to(dtype)
    rows, dy_rows = torch.randn(256, 1024, device=DEV).to(dtype), torch.randn(256, 1024, device=DEV).to(dtype)
    x, dy = rows.repeat(9, 1)[:2200].requires_grad_(True), dy_rows.repeat(9, 1)[:2200]
    y = layer(x)
    dx, = torch.autograd.grad(y, x, dy)
    w = dense_weight(layer.weight, layer.matrix.backward_indices, 1024).abs()
    unit, tiny = UNIT[dtype], 2.0**-24 if dtype == torch.float16 else 0.0
    for got, magnitude in ((y.detach().double(), rows.double().abs() @ w.t()), (dx.double(), dy_rows.double().abs() @ w)):
        bound = 2 * (1024 + 16) * 2.0**-23 * magnitude * (1 + unit) + 2 * tiny
        for tile in range(1, 9):
            part = got[256 * tile:256 * (tile + 1)]
            worst = (part - got[:len(part)]).abs() - bound[:len(part)] - 2 * unit * got[:len(part)].abs() * (1 + unit)
            assert worst.max().item() <= 0.0, (tile, worst.max().item())
