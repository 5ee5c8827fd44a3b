"""LayerNorm backward with both gradients from one pass (16-bit dy, rows of up to 4096 elements): edges of the columns a lane and a
wavefront hold, of the rows a workgroup takes at a time, several turns of its loop, and the sizes on either side of the rule."""
import pytest
import torch

from lean_transformer_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _backward(x, dy, res, w, stats, dx_dtype, workspace_rows=None):
    tokens, hidden = x.shape
    lib = nat.lib(dy.dtype)
    dx = torch.full((tokens, hidden), float("nan"), dtype=dx_dtype, device=DEV)
    dw, db = torch.full((hidden,), float("nan"), device=DEV), torch.full((hidden,), float("nan"), device=DEV)
    size = lib.lt_layernorm_backward_workspace_bytes(tokens, hidden) if workspace_rows is None else workspace_rows * 8 * hidden
    ws = nat.workspace(size, torch.device(DEV))
    ws.fill_(0xFF)
    nat.check(lib.lt_layernorm_backward(tokens, hidden, nat.dtype_code(x.dtype), nat.ptr(x), nat.ptr(stats), nat.ptr(w),
                                        nat.dtype_code(dy.dtype), nat.ptr(dy), nat.dtype_code(dx_dtype), nat.ptr(res), nat.ptr(dx),
                                        nat.ptr(dw), nat.ptr(db), nat.ptr(ws), size, nat.current_stream(dx.device)),
              "lt_layernorm_backward", lib)
    return dx, dw, db


def _inputs(tokens, hidden, x_dtype, dy_dtype, dx_dtype):
    g = torch.Generator(device=DEV).manual_seed(tokens + hidden)
    x = (torch.randn(tokens, hidden, generator=g, device=DEV) * 2 + 0.5).to(x_dtype)
    dy = torch.randn(tokens, hidden, generator=g, device=DEV).to(dy_dtype)
    res = torch.randn(tokens, hidden, generator=g, device=DEV).to(dx_dtype)
    w = torch.rand(hidden, generator=g, device=DEV) + 0.5
    xd = x.double()
    stats = torch.stack([xd.mean(-1), torch.rsqrt(xd.var(-1, unbiased=False) + 1e-5)], 1).float().contiguous()
    return x, dy, res, w, stats


def _check(x, dy, res, w, stats, got):
    dx, dw, db = got
    xh = (x.double() - stats[:, :1].double()) * stats[:, 1:].double()
    g = dy.double()
    dxh = g * w.double()
    ref = stats[:, 1:].double() * (dxh - dxh.mean(-1, keepdim=True) - xh * (dxh * xh).mean(-1, keepdim=True))
    if res is not None:
        ref = ref + res.double()
    # dx: a rounding to its type (half a unit in the last of 8 significant bits, of 11 in fp16) over fp32 arithmetic on values of order 1
    half_unit = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dx.dtype]
    assert ((dx.double() - ref).abs() <= half_unit * 1.01 * ref.abs() + 1e-5).all()
    # column sums: about 112 additions (rows of a lane, the groups of a workgroup, the partial rows), half a unit of 24 bits each
    for name, sums, terms in (("dweight", dw, g * xh), ("dbias", db, g)):
        bound = 8e-6 * terms.abs().sum(0) + 1e-6
        assert ((sums.double() - terms.sum(0)).abs() <= bound).all(), name


@pytest.mark.parametrize("tokens,hidden", [(1, 4), (17, 252), (300, 768), (5000, 1024), (15, 1028), (2500, 2048), (9, 2052),
                                           (1031, 3000), (1500, 4096), (70, 4100)])
@pytest.mark.parametrize("x_dtype,dy_dtype,dx_dtype", [(torch.float32, torch.bfloat16, torch.float32),
                                                       (torch.float32, torch.bfloat16, torch.bfloat16),
                                                       (torch.bfloat16, torch.bfloat16, torch.float32),
                                                       (torch.float16, torch.float16, torch.float16)])
@pytest.mark.parametrize("with_residual", [False, True])
def test_one_pass(tokens, hidden, x_dtype, dy_dtype, dx_dtype, with_residual):
    x, dy, res, w, stats = _inputs(tokens, hidden, x_dtype, dy_dtype, dx_dtype)
    res = res if with_residual else None
    _check(x, dy, res, w, stats, _backward(x, dy, res, w, stats, dx_dtype))


@pytest.mark.parametrize("partial_rows", [15, 17, 112, 127, 128, 129, 241])
def test_sums_of_any_number_of_partial_rows(partial_rows):
    """16 row lanes read eight partial rows ahead: around one turn of that, several, and a rest (68 columns: a column block and a bit)"""
    tensors = _inputs(16 * partial_rows, 68, torch.float32, torch.bfloat16, torch.float32)
    _check(*tensors, _backward(*tensors, torch.float32))


def test_scratch_for_the_two_kernels_alone_is_still_enough():
    tensors = _inputs(640, 1024, torch.float32, torch.bfloat16, torch.float32)
    _check(*tensors, _backward(*tensors, torch.float32, workspace_rows=10))  # (the one pass would take 40)


def test_a_row_of_nan_stays_in_its_row():
    x, dy, res, w, stats = _inputs(2100, 2048, torch.float32, torch.bfloat16, torch.float32)
    dy[7, 3] = float("nan")
    dx, dw, db = _backward(x, dy, res, w, stats, torch.float32)
    assert dx[7].isnan().all() and dw[3].isnan() and db[3].isnan()
    assert dx[:7].isfinite().all() and dx[8:].isfinite().all()
    assert dw.isnan().sum() == 1 and db.isnan().sum() == 1
