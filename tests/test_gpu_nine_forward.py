"""The 3x3 forward kernel (csrc/fwd_nine.hip) against the float64 oracle where its strips, rows, tiles and waves end: rows of one, two
and three columns, maps of one row, odd and even rows at stride 2, channels that give a wave no chunk or part of one, output channels
that fill no block -- with its statistics, its inference epilogue, bases of any
alignment and both storage types.  (Each number of waves and of positions per lane:
test_gpu_kernel_shapes; as an ordinary convolution and with the strided 1x1 layer beside it: test_gpu_resnet20, test_gpu_pair.)"""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, stride)
SHAPES = [(1, 1, 1, 1, 1, 1), (2, 9, 5, 1, 9, 1), (3, 33, 1, 2, 7, 1), (2, 8, 3, 3, 12, 1), (70, 17, 2, 5, 5, 1), (1, 264, 7, 7, 31, 1),
          (3, 130, 14, 14, 33, 1), (9, 24, 9, 33, 40, 1), (2, 70, 56, 55, 9, 1),                      # one position per lane
          (200, 7, 32, 29, 12, 1), (64, 16, 33, 35, 20, 1), (60, 30, 17, 17, 70, 1), (12, 64, 30, 32, 40, 1),   # two and four
          (1, 3, 1, 1, 2, 2), (2, 9, 5, 1, 9, 2), (2, 12, 1, 7, 5, 2), (5, 35, 2, 2, 3, 2), (4, 20, 18, 18, 18, 2), (4, 20, 17, 19, 18, 2),
          (64, 16, 32, 32, 32, 2), (130, 40, 9, 9, 40, 2), (40, 5, 21, 24, 70, 2)]


def _case(shape):
    return shape[:5] + (3, shape[5], 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matches_the_oracle(shape, dtype, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    s = shape[5]
    x, w, _ = make_case(*_case(shape))
    x = x.to(dtype)
    want = c_oracle.conv2d_fwd(x.float(), w, s, 1)
    xg, wg = x.to(gpu), w.to(gpu)
    y = adder.adder2d_function(xg, wg, s, 1)
    (assert_close if dtype == torch.float32 else _close_bf16)(y, want, f"forward {shape}")
    off = torch.empty(xg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(xg).copy_(xg)   # aligned to one element only
    assert torch.equal(adder.adder2d_function(off, wg, s, 1), y)
    if dtype == torch.float32:
        y2, stats = adder.adder2d_function_with_stats(xg, wg, s, 1)
        assert torch.equal(y2, y)
        tot = stats.sum(dim=1).cpu()
        assert torch.allclose(tot[:, 0], want.sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-3)
        assert torch.allclose(tot[:, 1], (want * want).sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-2)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_inference_epilogue(shape, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    N, Ci, H, W, Co, s = shape
    x, w, gy = (t.to(gpu) for t in make_case(*_case(shape)))
    y, res, out = torch.empty_like(gy), torch.randn_like(gy), torch.empty_like(gy)
    gamma, beta, mean, var = (torch.rand(Co, device=gpu) + 0.5 for _ in range(4))
    dims = (N, Ci, H, W, Co, 3, 3, s, 1, stream_ptr(x.device))
    assert lib.adder_conv2d_fwd_f32(ptr(x), ptr(w), ptr(y), *dims) == 0
    col = lambda t: t.view(1, -1, 1, 1)
    for residual, relu in ((None, 0), (res, 1)):
        assert lib.adder_conv2d_fwd_bn_eval_f32(ptr(x), ptr(w), ptr(out), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5,
                                                ptr(residual), relu, *dims) == 0
        want = (y - col(mean)) * torch.rsqrt(col(var) + 1e-5) * col(gamma) + col(beta)
        want = torch.relu(want + residual) if relu else want
        # a few roundings of values of y's size: 4 ulp
        assert torch.allclose(out, want, rtol=0, atol=4 * 2 ** -23 * (float(y.abs().max()) * 2 + 4))


@pytest.mark.parametrize("stride", [1, 2])
def test_infinities_and_nan_pass(stride, gpu):
    """What lies outside the map counts as zero whatever stands at the map's edge."""
    from addernetcuda_amd import adder
    x, w, _ = make_case(2, 9, 6, 7, 12, 3, stride, 1)
    x[0, 3, 0, 0], x[1, 8, 5, 6], x[1, 0, 2, 0], w[5, 2, 1, 1] = float("inf"), float("nan"), float("-inf"), float("-inf")
    y = adder.adder2d_function(x.to(gpu), w.to(gpu), stride, 1).cpu()
    cols = torch.nn.functional.pad(x, (1, 1, 1, 1)).unfold(2, 3, stride).unfold(3, 3, stride)   # (N, Ci, Ho, Wo, 3, 3)
    want = -(w.view(1, 12, 9, 1, 1, 3, 3) - cols.unsqueeze(1)).abs().sum((2, 5, 6))
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf())
