"""Thin products of a low-rank term: hid = x L1^T and g L2 of up to 64 columns, read out through a zero weight and an identity for the other
factor (the product with it is exact).  Rows around the 16-row tiles and the line between the two workgroup shapes, ranks around the 16-column
tiles, reductions around the 16-byte pieces and 64-k blocks.

Bound: fp32 accumulation of exact products, at most K + 16 additions each off by 2^-23 of the magnitudes it adds, and one rounding to 16 bits."""
import pytest
import torch

from lean_transformer_amd import _native as nat
from lean_transformer_amd.blocksparse.linear import GeneralizedLinear, GeneralizedMatrix

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(fan_in, fan_out, rank, dtype):
    layer = GeneralizedLinear(GeneralizedMatrix(fan_in, fan_out), adapter_dim=rank, bias=False).to(DEV).to(dtype)
    with torch.no_grad():
        layer.weight.zero_()
    return layer


def _check(got, a, b, dtype):
    ref, room = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    worst = (got.double() - ref).abs() - ((a.shape[1] + 16) * 2.0**-23 * room * 2 + unit * ref.abs() + 2.0**-24)
    assert worst.max().item() <= 0.0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank", [8, 16, 24, 32, 40, 64])
@pytest.mark.parametrize("tokens,k", [(65, 8), (80, 64), (127, 72), (1000, 1096), (4096, 64), (4097, 64), (8191, 136), (8192, 128), (8209, 200), (66, 2048), (300, 2040)])
def test_both_factors(dtype, rank, tokens, k):
    g = torch.Generator(device=DEV).manual_seed(tokens + k + rank)
    long = (torch.randn(tokens, k, generator=g, device=DEV) * 0.25).to(dtype)
    factor = torch.randn(k, rank, generator=g, device=DEV).to(dtype)
    eye = torch.eye(rank, device=DEV, dtype=dtype)
    lib = nat.lib(dtype)

    def thin(fn):
        lib.lt_profile_reset()
        lib.lt_profile_enable(1)
        out = fn()
        lib.lt_profile_enable(0)
        assert ("gemm_thin" in {e[0] for e in nat.profile_read(lib)}) == (rank <= 16 or tokens <= 8192)
        return out

    layer = _layer(k, rank, rank, dtype)
    with torch.no_grad():
        layer.adapter_first.copy_(factor.t())
        layer.adapter_second.copy_(eye)
        hid = thin(lambda: layer(long))
    _check(hid, long, factor, dtype)

    layer = _layer(rank, k, rank, dtype)
    with torch.no_grad():
        layer.adapter_first.copy_(eye)
        layer.adapter_second.copy_(factor)
    x = torch.zeros(tokens, rank, device=DEV, dtype=dtype, requires_grad=True)
    y = layer(x)
    g_hid, = thin(lambda: torch.autograd.grad(y, x, long))
    _check(g_hid, long, factor, dtype)


@pytest.mark.parametrize("tokens,k,rank", [(64, 64, 16), (8193, 3080, 16), (8193, 64, 24), (300, 2056, 40), (300, 4104, 24), (300, 64, 72), (300, 60, 16), (300, 64, 12)])
def test_neighbours_of_the_rule(tokens, k, rank):
    """products on the other side of each line, through the same layers"""
    g = torch.Generator(device=DEV).manual_seed(tokens + k + rank)
    long = (torch.randn(tokens, k, generator=g, device=DEV) * 0.25).bfloat16()
    factor = torch.randn(k, rank, generator=g, device=DEV).bfloat16()
    eye = torch.eye(rank, device=DEV, dtype=torch.bfloat16)
    layer = _layer(rank, k, rank, torch.bfloat16)
    with torch.no_grad():
        layer.adapter_first.copy_(eye)
        layer.adapter_second.copy_(factor)
    x = torch.zeros(tokens, rank, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    g_hid, = torch.autograd.grad(layer(x), x, long)
    _check(g_hid, long, factor, torch.bfloat16)


@pytest.mark.parametrize("tokens,thin", [(16384, True), (16385, False), (65536, False), (65537, True)])
def test_rows_of_the_rule(tokens, thin):
    """up to 16 columns: rows of one launch's workgroups, and more than 128 x 128 tiles run at once"""
    layer = _layer(64, 8, 16, torch.bfloat16)
    x = torch.randint(-2, 3, (tokens, 64), device=DEV).bfloat16()
    with torch.no_grad():
        layer.adapter_first.copy_(torch.eye(16, 64))
        layer.adapter_second.copy_(torch.eye(8, 16))
        lib = nat.lib(torch.bfloat16)
        lib.lt_profile_reset()
        lib.lt_profile_enable(1)
        y = layer(x)
        lib.lt_profile_enable(0)
    assert ("gemm_thin" in {e[0] for e in nat.profile_read(lib)}) == thin and torch.equal(y, x[:, :8])


def test_values_past_the_end_are_not_read_into_the_sums():
    """rows of the factor and of the activation behind the last one hold NaN in memory"""
    tokens, k, rank = 100, 72, 24
    whole = torch.full((tokens + 64, k), float("nan"), device=DEV, dtype=torch.bfloat16)
    whole[:tokens] = 1.0
    first = torch.full((rank + 64, k), float("nan"), device=DEV, dtype=torch.bfloat16)
    first[:rank] = 0.5
    second = torch.full((k + 64, rank), float("nan"), device=DEV, dtype=torch.bfloat16)
    second[:k] = 0.5
    layer = _layer(k, rank, rank, torch.bfloat16)
    layer.adapter_first.data, layer.adapter_second.data = first[:rank], torch.eye(rank, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        assert (layer(whole[:tokens]) == 36.0).all()
    layer = _layer(rank, k, rank, torch.bfloat16)
    layer.adapter_first.data, layer.adapter_second.data = torch.eye(rank, device=DEV, dtype=torch.bfloat16), second[:k]
    x = torch.zeros(tokens, rank, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    dx, = torch.autograd.grad(layer(x), x, whole[:tokens])
    assert (dx == 36.0).all()
