"""The any-shape GEMM kernel: fp32 operands as three bfloat16 planes, its tile heights (64 and 128 rows), vector and scalar fetches,
whole and ragged k-steps, split reductions, block-sparse walks over odd block sizes.

Bound on a result of fp32 operands: the six plane products are exact in fp32, so an element is a chain of at most 6 ceil(K / 16) + 4
fp32 accumulations (4 for the sum of the slices), each off by at most 2^-23 of the magnitudes it adds, plus the dropped products, at
most 2^-22 of |a| |b|:  |c - ref| <= (6 ceil(K / 16) + 6) 2^-23 (|a| |b|^T)."""
import pytest
import torch

from conftest import rel_err
from lean_transformer_amd import _native as nat
from test_gpu_kernels import _gemm, _operands

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(c, a, b, k):
    """a [m, k], b [n, k] on the GPU"""
    ref = a.double() @ b.double().t()
    bound = (6 * -(-k // 16) + 6) * 2.0**-23 * (a.double().abs() @ b.double().abs().t())
    worst = ((c.double() - ref).abs() - bound).max().item()
    assert worst <= 0.0, f"{worst:.3e} beyond the bound"
    return ref


@pytest.mark.parametrize("a_kmajor,b_kmajor", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (64, 128, 16), (65, 129, 17), (63, 127, 15), (130, 132, 48), (200, 260, 100),
                                   (5000, 1700, 36), (4100, 2048, 64)])
def test_fp32_any_shape_and_layout(a_kmajor, b_kmajor, m, n, k):
    """the last two have enough workgroups for 128-row tiles"""
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    c = _gemm(a if a_kmajor else a.t().contiguous(), b if b_kmajor else b.t().contiguous(), a_kmajor, b_kmajor, m, n, k,
              torch.float32, 1)
    _check(c, a, b, k)


@pytest.mark.parametrize("scale", [1.0, 2.0**100, 2.0**-90])
def test_fp32_split_is_exact(scale):
    """times the identity: every element comes back bit for bit, from the largest finite value down"""
    g = torch.Generator(device=DEV).manual_seed(1)
    a = torch.randn(130, 96, generator=g, device=DEV) * scale
    a[0, :4] = torch.tensor([torch.finfo(torch.float32).max, -torch.finfo(torch.float32).max, 0.0, 1 + 2.0**-23], device=DEV)
    eye = torch.eye(96, device=DEV)
    assert torch.equal(_gemm(a, eye, True, True, 130, 96, 96, torch.float32, 1), a)


def test_fp32_errors_do_not_add_up_over_rows():
    """a bias of the accumulation's rounding would grow with the number of rows in a column sum (a bias gradient): the sum of M
    independent errors is sqrt(M) times one of them; 4 times that leaves room for a bias of 6 % of the rms error at M = 4096"""
    g = torch.Generator(device=DEV).manual_seed(2)
    m, n, k = 4096, 768, 1536
    a, b = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    err = _gemm(a, b.t().contiguous(), True, False, m, n, k, torch.float32, 1).double() - a.double() @ b.double().t()
    assert err.sum(0).norm().item() <= 4 * err.norm().item()


def test_fp32_view_that_is_not_16_byte_aligned():
    """rows of an odd length behind an odd offset: element-wise fetches and stores"""
    g = torch.Generator(device=DEV).manual_seed(3)
    m, n, k = 70, 45, 33
    store = torch.randn(m * k + n * k + 2, generator=g, device=DEV)
    a, b = store[1:1 + m * k].view(m, k), store[1 + m * k:1 + m * k + n * k].view(n, k)
    out = torch.full((m * n + 9,), 7.0, device=DEV)
    c = out[1:1 + m * n].view(m, n)
    nat.check(nat.lib().lt_gemm(nat.LT_F32, m, n, k, a.data_ptr(), 1, b.data_ptr(), 1, nat.LT_F32, c.data_ptr(), 1,
                                nat.current_stream(c.device)), "lt_gemm")
    _check(c, a, b, k)
    assert out[0].item() == 7.0 and bool((out[1 + m * n:] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("a_kmajor,b_kmajor", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k", [(70, 45, 33), (129, 127, 31), (64, 128, 96), (4100, 2100, 72)])
def test_16_bit_operands(dtype, a_kmajor, b_kmajor, m, n, k):
    a, b, ref = _operands(m, n, k, a_kmajor, b_kmajor, dtype, seed=m + n + k)
    assert rel_err(_gemm(a, b, a_kmajor, b_kmajor, m, n, k, torch.float32, 1), ref) <= 1e-5


@pytest.mark.parametrize("a_kmajor,b_kmajor", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k", [(65, 129, 17), (4100, 2048, 64)])
def test_fp32_infinities_and_nans(a_kmajor, b_kmajor, m, n, k):
    """an infinity has no exact planes: the elements it reaches are computed again and come out as fp32 arithmetic gives them,
    infinite with the right sign, NaN where infinities of both signs or a zero meet; their neighbours are untouched"""
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, b = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    inf = float("inf")
    a[3, 5], a[8, k - 1], a[m - 1, 0], a[7, 1], a[7, 9], a[9, 2] = inf, -inf, inf, inf, -inf, float("nan")
    b[2, 5], b[n - 1, 5], b[4, 0] = 0.0, -inf, inf
    c = _gemm(a if a_kmajor else a.t().contiguous(), b if b_kmajor else b.t().contiguous(), a_kmajor, b_kmajor, m, n, k,
              torch.float32, 1)
    ref = (a.cpu().double() @ b.cpu().double().t()).to(DEV)
    assert torch.equal(c.isnan(), ref.isnan()) and torch.equal(c.isinf(), ref.isinf())
    assert torch.equal(c[c.isinf()].sign(), ref[ref.isinf()].sign().float())
    finite = ref.isfinite()
    assert (c.double() - ref)[finite].abs().max().item() <= 1e-4


def test_fp32_sums_of_zeros_are_positive():
    """odd rows are negated on their way through the matrix cores; their zeros come back as +0, as any sum from +0 does"""
    zeros, b = torch.zeros(70, 40, device=DEV), torch.randn(45, 40, device=DEV)
    c = _gemm(zeros, b, True, True, 70, 45, 40, torch.float32, 1)
    assert not bool(c.signbit().any()) and bool((c == 0).all())


@pytest.mark.parametrize("k", [1, 2, 3, 4, 16, 3072, 8192])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_fp32_sums_of_one_sign(k, sign):
    """no products are lost beside a large sum: 2-norm error at most that of K / 2 roundings to nearest (0.29 units of 2^-23 of a sum that
    grows evenly: sqrt(K / 2 / 3) of them), which is what adding two exact products at a time makes, and one rounding of the result"""
    g = torch.Generator(device=DEV).manual_seed(k)
    a, b = torch.randn(256, k, generator=g, device=DEV).abs(), sign * torch.randn(512, k, generator=g, device=DEV).abs()
    ref = a.double() @ b.double().t()
    err = _gemm(a, b, True, True, 256, 512, k, torch.float32, 1).double() - ref
    assert (err.norm() / ref.norm()).item() <= 0.29 * 2.0**-23 * (1 + (k / 6) ** 0.5)
    if k == 1:  # one rounding, of a sum that the planes give to 2^-30
        assert (err.abs() / ref.abs()).max().item() <= 2.0**-24 * (1 + 2.0**-6)
