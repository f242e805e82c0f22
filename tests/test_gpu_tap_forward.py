"""The 1x1 forward kernel (csrc/fwd_tap.hip) against the float64 oracle where its strips, tiles and waves end: planes of 1
to 4 positions and of no whole strips, channels that give a wave no chunk or part of one, output channels that fill no block, one,
two and four positions per lane (with each number of waves: test_gpu_kernel_shapes) -- with its statistics, its inference epilogue, bases of any alignment and both storage types."""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co): one position per lane, two, four; planes of whole strips and not
SHAPES = [(1, 64, 1, 1, 8), (3, 64, 1, 2, 9), (70, 68, 1, 3, 5), (65, 64, 2, 2, 1), (5, 128, 7, 7, 18), (2, 132, 13, 1, 1), (1, 1028, 5, 5, 7),
          (16, 128, 20, 20, 64), (9, 516, 9, 9, 130), (300, 64, 7, 7, 64), (40, 256, 15, 15, 72), (64, 260, 14, 14, 64), (33, 76, 32, 32, 24)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matches_the_oracle(shape, dtype, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    x, w, _ = make_case(*shape, 1, 1, 0)
    x = x.to(dtype)
    want = c_oracle.conv2d_fwd(x.float(), w, 1, 0)
    xg, wg = x.to(gpu), w.to(gpu)
    y = adder.adder2d_function(xg, wg, 1, 0)
    (assert_close if dtype == torch.float32 else _close_bf16)(y, want, f"forward {shape}")
    # a base aligned to one element only
    off = torch.empty(xg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(xg).copy_(xg)
    assert torch.equal(adder.adder2d_function(off, wg, 1, 0), y)
    if dtype == torch.float32:
        y2, stats = adder.adder2d_function_with_stats(xg, wg, 1, 0)
        assert torch.equal(y2, y)
        tot = stats.sum(dim=1).cpu()
        assert torch.allclose(tot[:, 0], want.sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-3)
        assert torch.allclose(tot[:, 1], (want * want).sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-2)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_inference_epilogue(shape, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    N, Ci, H, W, Co = shape
    x, w, _ = (t.to(gpu) for t in make_case(*shape, 1, 1, 0))
    y, res, out = torch.empty(N, Co, H, W, device=gpu), torch.randn(N, Co, H, W, device=gpu), torch.empty(N, Co, H, W, device=gpu)
    gamma, beta, mean, var = (torch.rand(Co, device=gpu) + 0.5 for _ in range(4))
    dims = (N, Ci, H, W, Co, 1, 1, 1, 0, stream_ptr(x.device))
    assert lib.adder_conv2d_fwd_f32(ptr(x), ptr(w), ptr(y), *dims) == 0
    col = lambda t: t.view(1, -1, 1, 1)
    for residual, relu in ((None, 0), (res, 1)):
        assert lib.adder_conv2d_fwd_bn_eval_f32(ptr(x), ptr(w), ptr(out), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5,
                                                ptr(residual), relu, *dims) == 0
        want = (y - col(mean)) * torch.rsqrt(col(var) + 1e-5) * col(gamma) + col(beta)
        want = torch.relu(want + residual) if relu else want
        # a few roundings of values of y's size: 4 ulp
        assert torch.allclose(out, want, rtol=0, atol=4 * 2 ** -23 * (float(y.abs().max()) * 2 + 4))


def test_infinities_and_nan_pass(gpu):
    from addernetcuda_amd import adder
    x, w, _ = make_case(2, 64, 7, 7, 12, 1, 1, 0)
    x[0, 3, 0, 0], x[1, 63, 6, 6], w[5, 2] = float("inf"), float("nan"), float("-inf")
    y = adder.adder2d_function(x.to(gpu), w.to(gpu), 1, 0).cpu()
    want = -(w.view(1, 12, 64, 1, 1) - x.unsqueeze(1)).abs().sum(2)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf())


# (N, Ci, H, W, Co, stride): channels below, at and beside whole groups and chunks, with and without a stride; planes whose sampled positions are
# no whole strips, whose last row or column is not read, and tiles that span several images
ANY = [(1, 1, 1, 1, 1, 1), (3, 3, 5, 7, 9, 1), (5, 17, 9, 9, 10, 1), (68, 33, 7, 7, 19, 1), (4, 373, 13, 16, 9, 1), (2, 131, 9, 10, 33, 1), (40, 30, 32, 32, 24, 1),
       (30, 24, 30, 30, 9, 1), (1, 16, 32, 32, 32, 2), (20, 6, 29, 29, 18, 2), (1, 5, 1, 1, 3, 2), (9, 68, 3, 3, 40, 2), (2, 130, 7, 9, 17, 3), (70, 40, 13, 13, 64, 2),
       (33, 68, 27, 28, 40, 2), (20, 263, 14, 14, 130, 2), (40, 64, 20, 21, 60, 3), (30, 20, 61, 62, 9, 2), (64, 12, 60, 61, 24, 3)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", ANY, ids=str)
def test_any_channels_and_strides(shape, dtype, gpu):
    from addernetcuda_amd import adder
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    from oracle import c_oracle
    N, Ci, H, W, Co, s = shape
    x, w, gy = make_case(N, Ci, H, W, Co, 1, s, 0)
    x = x.to(dtype)
    want = c_oracle.conv2d_fwd(x.float(), w, s, 0)
    xg, wg = x.to(gpu), w.to(gpu)
    y = adder.adder2d_function(xg, wg, s, 0)
    (assert_close if dtype == torch.float32 else _close_bf16)(y, want, f"forward {shape}")
    off = torch.empty(xg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(xg).copy_(xg)   # aligned to one element only
    assert torch.equal(adder.adder2d_function(off, wg, s, 0), y)
    if dtype != torch.float32:
        return
    y2, stats = adder.adder2d_function_with_stats(xg, wg, s, 0)
    assert torch.equal(y2, y)
    assert (stats is None) == (s > 2 and (Ci < 64 or Ci % 4 != 0))   # (never offered for those)
    if stats is not None:
        tot = stats.sum(dim=1).cpu()
        assert torch.allclose(tot[:, 0], want.sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-3)
        assert torch.allclose(tot[:, 1], (want * want).sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-2)
    out, res = torch.empty_like(y), torch.randn_like(y)
    gamma, beta, mean, var = (torch.rand(Co, device=gpu) + 0.5 for _ in range(4))
    assert lib.adder_conv2d_fwd_bn_eval_f32(ptr(xg), ptr(wg), ptr(out), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5, ptr(res), 1,
                                            N, Ci, H, W, Co, 1, 1, s, 0, stream_ptr(xg.device)) == 0
    col = lambda t: t.view(1, -1, 1, 1)
    want = torch.relu((y - col(mean)) * torch.rsqrt(col(var) + 1e-5) * col(gamma) + col(beta) + res)
    # a few roundings of values of y's size: 4 ulp
    assert torch.allclose(out, want, rtol=0, atol=4 * 2 ** -23 * (float(y.abs().max()) * 2 + 4))
