"""The sigmoid of the 16-bit activations over every 16-bit input, down to the smallest normal result: silu(-88) is -5e-37, which a
reciprocal that flushes subnormal results returns as 0.

Bound: half a unit in the last place of the stored type (8 significant bits: 2^-8 of the value; 11: 2^-11), and 2^-15 for the fp32 evaluation (the exponential's argument, up to 127 in base
2, is rounded to 2^-24 of itself: 2^-17; the rest is a few units of 2^-24)."""
import pytest
import torch

from lean_transformer_amd import _native as nat
from lean_transformer_amd.utils import ACT_KINDS
from oracle import ffn as offn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("act,slope", [("silu", 1.0), ("quick_gelu", 1.702)])
@pytest.mark.parametrize("dtype,unit", [(torch.bfloat16, 2.0**-8), (torch.float16, 2.0**-11)])
def test_every_input(act, slope, dtype, unit):
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).view(64, 1024).to(DEV)
    got = torch.empty_like(x)
    lib = nat.lib(dtype)
    nat.check(lib.lt_activation_forward(64, 1024, 0, ACT_KINDS[act], nat.dtype_code(dtype), nat.ptr(x), nat.ptr(got),
                                        nat.current_stream(x.device)), "lt_activation_forward", lib)
    ref = offn.act_forward(act, x.double())
    finite = (-slope * x.double()).exp() < torch.finfo(torch.float32).max  # (beyond it the fp32 sigmoid is 0)
    normal = x.isfinite() & finite & (ref.abs() >= torch.finfo(dtype).smallest_normal)
    assert ((got.double() - ref).abs() - (unit + 2.0**-15) * ref.abs())[normal].max().item() <= 0.0
    assert bool((got[x == -float("inf")].isnan()).all()) and bool((got[x == float("inf")] == float("inf")).all())
