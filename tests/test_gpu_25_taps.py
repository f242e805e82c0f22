"""5x5 layers (csrc/fwd_nine.hip with 25 taps) against the float64 oracle where strips, tiles, pairs of columns and waves end: maps of one row or
column, rows one longer than whole strips, rows whose last strip is moved back, even and odd rows at stride 2, channels that
give a wave none -- with the inference epilogue, bases of any alignment and both storage types."""
import pytest
import torch

from tests.util import make_case, assert_close, fwd_kernel, grad_x_kernel, NINE
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co)
SHAPES = [(1, 1, 1, 1, 1), (3, 5, 1, 2, 7), (2, 7, 3, 4, 9), (4, 3, 4, 5, 6), (2, 9, 6, 7, 17), (70, 8, 9, 9, 21), (40, 13, 17, 18, 30), (30, 20, 14, 15, 33),
          (64, 40, 16, 16, 24), (9, 67, 21, 20, 41), (9, 66, 20, 21, 40), (33, 9, 27, 23, 20)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(shape, stride, dtype, gpu):
    from addernetcuda_amd import adder
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    from oracle import c_oracle
    N, Ci, H, W, Co = shape
    x, w, _ = make_case(*shape, 5, stride, 2)
    x = x.to(dtype)
    want = c_oracle.conv2d_fwd(x.float(), w, stride, 2)
    xg, wg = x.to(gpu), w.to(gpu)
    y = adder.adder2d_function(xg, wg, stride, 2)
    (assert_close if dtype == torch.float32 else _close_bf16)(y, want, f"forward {shape}")
    off = torch.empty(xg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(xg).copy_(xg)   # aligned to one element only
    assert torch.equal(adder.adder2d_function(off, wg, stride, 2), y)
    if dtype != torch.float32:
        return
    out, res = torch.empty_like(y), torch.randn_like(y)
    gamma, beta, mean, var = (torch.rand(Co, device=gpu) + 0.5 for _ in range(4))
    assert lib.adder_conv2d_fwd_bn_eval_f32(ptr(xg), ptr(wg), ptr(out), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5, ptr(res), 1,
                                            N, Ci, H, W, Co, 5, 5, stride, 2, stream_ptr(xg.device)) == 0
    col = lambda t: t.view(1, -1, 1, 1)
    want = torch.relu((y - col(mean)) * torch.rsqrt(col(var) + 1e-5) * col(gamma) + col(beta) + res)
    # a few roundings of values of y's size: 4 ulp
    assert torch.allclose(out, want, rtol=0, atol=4 * 2 ** -23 * (float(y.abs().max()) * 2 + 4))


def test_infinities_and_nan_pass(gpu):
    from addernetcuda_amd import adder
    x, w, _ = make_case(2, 9, 12, 14, 12, 5, 1, 2)
    x[0, 3, 0, 0], x[1, 8, 11, 13], w[5, 2, 1, 1] = float("inf"), float("nan"), float("-inf")
    y = adder.adder2d_function(x.to(gpu), w.to(gpu), 1, 2).cpu()
    u = torch.nn.functional.unfold(x, 5, padding=2)
    want = -(w.view(1, 12, -1, 1) - u.unsqueeze(1)).abs().sum(2).view_as(y)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf())


# 4 x 2 and 4 x 1 results per lane with one to eight waves, rows of an odd length, more than 100 output channels; the last two stay in tiles
GRAD_X = SHAPES + [(40, 33, 16, 18, 12), (64, 40, 10, 10, 40), (9, 30, 22, 26, 131), (33, 40, 16, 16, 30), (70, 64, 16, 16, 24), (40, 64, 8, 32, 12)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", GRAD_X, ids=str)
def test_input_gradient(shape, dtype, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    x, w, gy = make_case(*shape, 5, 1, 2)
    x, gy = x.to(dtype), gy.to(dtype)
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, 1, 2)
    for base in (0, 1):   # aligned, and aligned to one element only
        g = torch.empty(gy.numel() + 1, dtype=dtype, device=gpu)[base:base + gy.numel()].view(gy.shape).copy_(gy)
        xg = x.to(gpu).requires_grad_(True)
        adder.adder2d_function(xg, w.to(gpu), 1, 2).backward(g)
        (assert_close if dtype == torch.float32 else _close_bf16)(xg.grad, want, f"grad_x {shape}, base {base}")


@pytest.mark.parametrize("shape", [(2, 7, 5, 6, 9), (64, 40, 10, 10, 40), (70, 64, 16, 16, 24), (2, 1, 9, 9, 4)], ids=str)
def test_second_gradient(shape, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims
    x, w, gy = (t.to(gpu) for t in make_case(*shape, 5, 1, 2))
    gadd, gx, out = torch.randn_like(x), torch.empty_like(x), torch.empty_like(x)
    dims, _, _ = conv_dims(x.shape, w.shape, 1, 2)
    st = stream_ptr(x.device)
    assert lib.adder_conv2d_bwd_f32(ptr(gy), ptr(x), ptr(w), ptr(gx), None, 0.0, None, 0, *dims, st) == 0
    rc = lib.adder_conv2d_bwd_add_f32(ptr(gy), ptr(x), ptr(w), ptr(gadd), ptr(out), None, 0.0, None, 0, *dims, st)
    if shape[1] >= 2:
        assert rc == 0 and torch.equal(out, gx + gadd)
    else:
        assert rc == -7   # one channel never had one


# Rows whose strips start a column earlier, so that no pair of columns beside one is half inside the row: four positions per lane on rows of whole strips and
# one column, two on rows of an odd length (from seven columns on)
ODD_ROWS = [(100, 12, 20, 9, 41), (100, 13, 11, 13, 41), (40, 20, 17, 17, 30), (60, 9, 14, 21, 41), (9, 41, 20, 37, 41), (16, 75, 17, 29, 21)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", ODD_ROWS, ids=str)
def test_rows_of_whole_strips_and_one_column(shape, dtype, gpu):
    assert fwd_kernel(shape + (5, 1, 2))[:3] == (NINE, 4, 4)
    test_forward(shape, 1, dtype, gpu)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", ODD_ROWS + [(33, 30, 13, 7, 41), (33, 21, 9, 11, 60), (16, 20, 14, 23, 131)], ids=str)
def test_input_gradient_of_odd_rows(shape, dtype, gpu):
    assert grad_x_kernel(shape + (5, 1, 2), dtype == torch.bfloat16)[:3] == (NINE, 4, 2)
    test_input_gradient(shape, dtype, gpu)
