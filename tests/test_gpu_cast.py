"""lt_cast: fp32 tensors to 16 bits in one launch, bit for bit what torch's conversion gives (NaN payloads aside), for sizes around a lane's 8
elements and a workgroup's 2048, odd addresses, more tensors than one launch holds, and tensors it leaves to torch."""
import pytest
import torch

from lean_transformer_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sizes", [[1], [7, 8, 9], [2047, 2048, 2049, 3], [5000000, 1, 4096], list(range(1, 20))])
@pytest.mark.parametrize("odd", [False, True])
def test_cast(dtype, sizes, odd):
    g = torch.Generator(device=DEV).manual_seed(sum(sizes))
    tensors = []
    for i, n in enumerate(sizes):
        flat = torch.randn(n + 1, generator=g, device=DEV) * 10.0 ** (i % 9 - 4)
        t = flat[1:] if odd else flat[:n]
        t[0] = [float("inf"), -0.0, 1e-42, float("nan"), 65519.9][i % 5]
        tensors.append(t)
    out = nat.cast_all([*tensors, None], dtype, DEV)
    assert out[-1] is None
    for t, o in zip(tensors, out):
        ref = t.to(dtype)
        assert o.dtype == dtype and o.shape == t.shape
        same = (o.view(torch.int16) == ref.view(torch.int16)) | (o.isnan() & ref.isnan())
        assert same.all()


def test_others_are_left_to_torch():
    a = torch.randn(6, 10, device=DEV)
    half = a.bfloat16()
    out = nat.cast_all([a.t(), half, a[:0], a], torch.bfloat16, DEV)
    assert torch.equal(out[0], a.t().contiguous().bfloat16()) and out[0].is_contiguous()
    assert out[1].data_ptr() == half.data_ptr() and out[2].shape == (0, 10)
    assert nat.cast_all([a], torch.float32, DEV)[0].data_ptr() == a.data_ptr()


def test_a_tensor_in_pieces():
    """2^30 elements are one piece of a launch"""
    n = (1 << 30) + 2051
    t = torch.arange(n, device=DEV, dtype=torch.int32).bitwise_and_(0xffff).float()
    out, = nat.cast_all([t], torch.bfloat16, DEV)
    for part in (slice(0, 4096), slice((1 << 30) - 4096, n)):
        assert torch.equal(out[part], t[part].bfloat16())
    assert torch.equal(out[::4097], t[::4097].bfloat16())
