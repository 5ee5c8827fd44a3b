"""A product and its low-rank term in one launch, on every kernel that takes two k-segments: lengths that are and are not multiples
of the 64-wide k-step and of the 8-element piece, either segment the ragged one.

Bound: fp32 accumulation of exact products of 16-bit elements, at most K + 16 additions each off by 2^-23 of the magnitudes it adds."""
import pytest
import torch

from lean_transformer_amd import _native as nat
from test_gpu_kernels import _kernel_tags

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def two_segments(dtype, m, n, k0, k1, a_kmajor, b_kmajor, force, seed=0):
    """(result, float64 reference, |a| |b|^T) of a random problem"""
    g = torch.Generator(device=DEV).manual_seed(seed + k0 + k1)
    pairs = [(torch.randn(m, k, generator=g, device=DEV).to(dtype), torch.randn(n, k, generator=g, device=DEV).to(dtype))
             for k in (k0, k1)]
    held = [(a if a_kmajor else a.t().contiguous(), b if b_kmajor else b.t().contiguous()) for a, b in pairs]
    c = torch.full((m, n), float("nan"), device=DEV)
    lib = nat.lib(dtype)
    (a0, b0), (a1, b1) = held
    nat.check(lib.lt_gemm_two_segments(nat.dtype_code(dtype), m, n, k0, nat.ptr(a0), nat.ptr(b0), k1, nat.ptr(a1), nat.ptr(b1),
                                       int(a_kmajor), int(b_kmajor), nat.LT_F32, nat.ptr(c), force,
                                       nat.current_stream(c.device)), "lt_gemm_two_segments", lib)
    ref = sum(a.double() @ b.double().t() for a, b in pairs)
    return c, ref, sum(a.double().abs() @ b.double().abs().t() for a, b in pairs)


@pytest.mark.parametrize("a_kmajor,b_kmajor", [(True, True), (True, False)])
@pytest.mark.parametrize("k0,k1", [(64, 64), (72, 64), (8, 128), (200, 64), (200, 72), (128, 8), (1000, 128)])
@pytest.mark.parametrize("force", [2, 3])
def test_tiled_kernels(a_kmajor, b_kmajor, k0, k1, force):
    """2: the register-staged kernel; 3: the copy-based one"""
    (c, ref, mag), tags = _kernel_tags(lambda: two_segments(torch.bfloat16, 300, 512, k0, k1, a_kmajor, b_kmajor, force))
    assert all(t.startswith("gemm_bf16_n") for t in tags), tags
    assert ((c.double() - ref).abs() - (k0 + k1 + 16) * 2.0**-23 * mag).max().item() <= 0.0


@pytest.mark.parametrize("a_kmajor,b_kmajor", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("dtype,k0,k1", [(torch.float32, 768, 34), (torch.float32, 96, 33), (torch.float32, 33, 96),
                                         (torch.bfloat16, 128, 65), (torch.bfloat16, 192, 97), (torch.bfloat16, 65, 192)])
@pytest.mark.parametrize("m,n", [(70, 45), (4100, 2100)])
def test_any_shape_kernel(dtype, k0, k1, a_kmajor, b_kmajor, m, n):
    """whole steps run from the first segment into the second, whose rows are not 16-byte aligned (rank 34 in fp32, 65 in 16 bits):
    it must be fetched element by element, and the other way round; both tile heights"""
    c, ref, mag = two_segments(dtype, m, n, k0, k1, a_kmajor, b_kmajor, 1)
    k = k0 + k1
    bound = 2.0**-23 * ((6 * (-(-k // 16) + 1) + 6) if dtype == torch.float32 else k + 16)  # (fp32: see test_gpu_any_shape.py)
    assert ((c.double() - ref).abs() - bound * mag).max().item() <= 0.0
