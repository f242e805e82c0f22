"""The input-gradient kernel of 3x3 / stride-1 layers (csrc/grad_x_nine.hip) against the float64 oracle where its strips, tiles, groups
of channels and waves end: rows that are shorter than a strip or whose last strip is moved back, input channels that do not fill a
group, output channels that end inside a chunk or give a wave none, one to eight waves -- with bases
of any alignment and both storage types; and with the BatchNorm link, which gives the plain kernel's bits.  (Each of its shapes in both forms:
test_gpu_kernel_shapes.)"""
import ctypes

import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co): 4 channels x 1 position with one to eight waves; 8 x 4 in two instructions a term
SHAPES = [(1, 4, 1, 1, 1), (3, 5, 1, 2, 7), (70, 9, 1, 3, 8), (2, 7, 5, 4, 9), (1, 3, 9, 9, 17), (9, 65, 7, 7, 129), (64, 17, 8, 8, 12),
          (60, 70, 17, 13, 16), (16, 67, 21, 19, 32), (9, 67, 21, 20, 40), (9, 67, 21, 20, 136),
          (40, 61, 33, 30, 5), (40, 70, 31, 29, 16), (30, 57, 21, 22, 30), (20, 67, 21, 18, 37), (20, 66, 21, 18, 131)]


def _grad_x(x, w, gy):
    from addernetcuda_amd import adder
    xg = x.clone().requires_grad_(True)
    adder.adder2d_function(xg, w, 1, 1).backward(gy)
    return xg.grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matches_the_oracle(shape, dtype, gpu):
    from oracle import c_oracle
    x, w, gy = make_case(*shape, 3, 1, 1)
    x, gy = x.to(dtype), gy.to(dtype)
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, 1, 1)
    xg, wg, gyg = x.to(gpu), w.to(gpu), gy.to(gpu)
    got = _grad_x(xg, wg, gyg)
    (assert_close if dtype == torch.float32 else _close_bf16)(got, want, f"grad_x {shape}")
    off = torch.empty(gyg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(gyg).copy_(gyg)   # aligned to one element only
    assert torch.equal(_grad_x(xg, wg, off), got)


# (links are offered for whole groups of four positions per row: 4 x 1, 8 x 2 and 8 x 4, one to eight waves, two instructions a term and three)
LINKED = [(2, 9, 3, 4, 7), (16, 19, 8, 8, 130), (60, 70, 17, 12, 16), (9, 68, 21, 20, 40), (40, 60, 33, 32, 5), (30, 57, 21, 20, 30),
          (20, 67, 21, 20, 131), (260, 9, 16, 16, 9), (130, 9, 32, 32, 9),
          (300, 30, 13, 16, 5), (300, 263, 3, 4, 11), (300, 130, 3, 4, 19), (60, 263, 3, 4, 41), (200, 263, 3, 4, 19), (200, 130, 3, 4, 41), (130, 5, 28, 28, 150)]


@pytest.mark.parametrize("shape", LINKED, ids=str)
def test_link_and_second_gradient_leave_the_bits(shape, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, BnLinks, bwd_bn_slots, conv_dims
    N, Ci, H, W, Co = shape
    x, w, gy = (t.to(gpu) for t in make_case(*shape, 3, 1, 1))
    x = torch.relu(x)
    gadd, bn_x, gx, out = torch.randn_like(x), torch.randn_like(x), torch.empty_like(x), torch.empty_like(x)
    mean, rstd = torch.randn(Ci, device=gpu), torch.rand(Ci, device=gpu) + 0.5
    dims, _, _ = conv_dims(x.shape, w.shape, 1, 1)
    slots, st = bwd_bn_slots(dims), stream_ptr(x.device)
    assert slots > 0
    assert lib.adder_conv2d_bwd_f32(ptr(gy), ptr(x), ptr(w), ptr(gx), None, 0.0, None, 0, *dims, st) == 0
    part = torch.full((Ci, slots, 2), float("nan"), device=gpu)
    links = BnLinks(None, None, None, ptr(bn_x), ptr(mean), ptr(rstd), ptr(part), slots, 1)
    assert lib.adder_conv2d_bwd_bn_f32(ptr(gy), ptr(x), ptr(w), ptr(gadd), ptr(out), None, 0.0, None, 0, *dims,
                                       ctypes.byref(links), st) == 0
    want = (gx + gadd) * (x > 0)
    assert torch.equal(out, want)
    xhat = (bn_x.double() - mean.double().view(1, -1, 1, 1)) * rstd.double().view(1, -1, 1, 1)
    sums = torch.stack([want.double().sum((0, 2, 3)), (want.double() * xhat).sum((0, 2, 3))], 1)
    scale = max(1.0, float(sums.abs().max()))
    assert_close(part.double().sum(1) / scale, sums / scale, "partial sums", rtol=1e-5, atol=1e-5)
