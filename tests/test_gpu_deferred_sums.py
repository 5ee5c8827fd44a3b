"""Sums that wait for one launch at the end of a backward pass: split weight and low-rank gradients, bias gradients, in room for all of
them, for some of them, and where nothing is split."""
import pytest
import torch

from lean_transformer_amd import _native as nat
from lean_transformer_amd.blocksparse.linear import GeneralizedMatrix, GeneralizedLinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


CASES = [
    (1, 8, 8, 0, True),          # nothing split, one column sum
    (257, 64, 72, 8, True),      # one tile a product
    (4099, 768, 320, 16, True),  # every gradient split, all of them wait
    (4099, 768, 320, 16, False),
    (4096, 1536, 2048, 64, True),   # a weight gradient too large to wait, summed at once, beside low-rank ones that wait
    (2051, 1003, 517, 5, True),     # sizes off every tile: the any-shape kernel's splits
]


@pytest.mark.parametrize("tokens,fan_in,fan_out,rank,bias", CASES)
@pytest.mark.parametrize("compute", ["autocast", "fp32"])
def test_gradients_summed_at_the_end(tokens, fan_in, fan_out, rank, bias, compute):
    torch.manual_seed(tokens + fan_in)
    layer = GeneralizedLinear(GeneralizedMatrix(fan_in, fan_out), adapter_dim=rank, bias=bias).to(DEV)
    with torch.no_grad():
        for p in layer.parameters():
            p.copy_(torch.randn_like(p).bfloat16() * 0.125)
    x = torch.randn(tokens, fan_in, device=DEV).bfloat16().float().requires_grad_(True)
    dy = torch.randn(tokens, fan_out, device=DEV).bfloat16().float()
    half = compute == "autocast"
    with torch.autocast("cuda", torch.bfloat16, enabled=half):
        y = layer(x)
    names, params = zip(*layer.named_parameters())
    first = torch.autograd.grad(y, params, dy.to(y.dtype), retain_graph=True)
    again = torch.autograd.grad(y, params, dy.to(y.dtype))
    xd, dyd = x.detach().double(), dy.double()
    for name, g, g2 in zip(names, first, again):
        assert torch.equal(g, g2), name
        if name.endswith("weight"):  # exact operands, fp32 sums: the worst case of a sum over the tokens
            ref, room = dyd.t() @ xd, dyd.abs().t() @ xd.abs()
        elif name == "bias":
            ref, room = dyd.sum(0), dyd.abs().sum(0)
        else:
            r1, r2 = layer.adapter_first.detach().double(), layer.adapter_second.detach().double()
            hid, g_hid = xd @ r1.t(), dyd @ r2
            pair = (dyd, hid) if name == "adapter_second" else (g_hid, xd)
            ref, room = pair[0].t() @ pair[1], pair[0].abs().t() @ pair[1].abs()
            if half:  # the other factor was rounded to bfloat16 (2^-9 of each term)
                assert ((g.double() - ref).abs() <= 2.0**-8 * room + 1e-30).all(), name
                continue
        assert ((g.double() - ref).abs() <= (tokens + fan_in + 64) * 2.0**-23 * room + 1e-30).all(), name


def check_whole_numbers(tokens, fan_in, fan_out, rank, bias, compute):
    """Gradients of whole numbers, and one-hot low-rank factors, whose products are columns of x and dy: every sum is
    exact (below 2^24), in any order, and none may lack a token.  Returns the launches of the backward pass by their tags."""
    torch.manual_seed(tokens + fan_out)
    layer = GeneralizedLinear(GeneralizedMatrix(fan_in, fan_out), adapter_dim=rank, bias=bias).to(DEV)
    x = torch.randint(-3, 4, (tokens, fan_in), device=DEV).float()
    dy = torch.randint(-3, 4, (tokens, fan_out), device=DEV).float()
    x[-1].abs_().add_(1.0)  # (the last token is in every sum)
    dy[-1].abs_().add_(1.0)
    expected = {"weight": dy.double().t() @ x.double(), "bias": dy.double().sum(0)}
    if rank:
        of_x, of_dy = torch.randperm(fan_in, device=DEV)[:rank], torch.randperm(fan_out, device=DEV)[:rank]
        one_hot = torch.nn.functional.one_hot
        with torch.no_grad():
            layer.adapter_first.copy_(one_hot(of_x, fan_in))
            layer.adapter_second.copy_(one_hot(of_dy, fan_out).t())
        expected["adapter_second"] = dy.double().t() @ x.double()[:, of_x]
        expected["adapter_first"] = dy.double()[:, of_dy].t() @ x.double()
    with torch.autocast("cuda", torch.bfloat16, enabled=compute == "autocast"):
        y = layer(x)
    names, params = zip(*layer.named_parameters())
    lib = nat.lib(torch.bfloat16)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    grads = torch.autograd.grad(y, params, dy.to(y.dtype))
    lib.lt_profile_enable(0)
    for name, g in zip(names, grads):
        assert g.dtype == torch.float32 and torch.equal(g.double(), expected[name.split(".")[-1]]), name
    return {tag: n for tag, n, *_ in nat.profile_read(lib)}


@pytest.mark.parametrize("tokens,fan_in,fan_out,rank,bias", CASES)
@pytest.mark.parametrize("compute", ["autocast", "fp32"])
def test_no_token_is_lost(tokens, fan_in, fan_out, rank, bias, compute):
    check_whole_numbers(tokens, fan_in, fan_out, rank, bias, compute)


def test_partial_results_that_do_not_all_fit():
    """split results take turns in the memory that holds the largest of them: the weight gradient's four slices (8 MiB) fill it, the low-rank
    pair's wait behind a first sum"""
    torch.manual_seed(0)
    layer = GeneralizedLinear(GeneralizedMatrix(512, 2048, "pixelfly(block_size=64, stretch=False)", 8)).to(DEV).bfloat16()
    x, dy = torch.randn(4096, 512, device=DEV, dtype=torch.bfloat16), torch.randn(4096, 2048, device=DEV, dtype=torch.bfloat16)
    y = layer(x)
    weight, pair = layer.matrix.weight, [layer.matrix.lowrank_first, layer.matrix.lowrank_second]
    lib = nat.lib(torch.bfloat16)
    lib.lt_profile_reset()
    lib.lt_profile_enable(1)
    together = torch.autograd.grad(y, [weight, *pair, layer.bias], dy, retain_graph=True)
    lib.lt_profile_enable(0)
    launches = {tag: n for tag, n, *_ in nat.profile_read(lib)}
    assert launches["splitk_reduce"] == 2, launches
    assert torch.equal(together[0], torch.autograd.grad(y, weight, dy, retain_graph=True)[0])
    for a, b in zip(together[1:], torch.autograd.grad(y, [*pair, layer.bias], dy)):
        assert torch.equal(a, b)
