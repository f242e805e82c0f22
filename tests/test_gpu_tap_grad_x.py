"""The input-gradient kernel of 1x1 / stride-1 layers (csrc/grad_x_tap.hip) against the float64 oracle where its strips, tiles, groups
of channels and waves end: planes of one to three positions and of an odd number, input channels that shift the last group, output
channels that end inside a group of four or give a wave no chunk -- with a second gradient, bases
of any alignment and both storage types; and with the BatchNorm link, which gives the plain kernel's bits.
(Each of its shapes in both forms: test_gpu_kernel_shapes.)"""
import ctypes

import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co): 8 channels x 1 position, then 16 x 2 with one to eight waves
SHAPES = [(1, 64, 1, 1, 48), (3, 65, 1, 2, 49), (70, 66, 1, 3, 51), (1, 64, 7, 7, 1030), (2, 127, 13, 1, 130), (5, 79, 9, 9, 64),
          (37, 67, 9, 9, 1027), (64, 72, 14, 14, 48), (40, 270, 7, 7, 129), (30, 100, 21, 21, 50), (160, 65, 21, 21, 50), (40, 80, 33, 32, 65)]


def _grad_x(x, w, gy):
    from addernetcuda_amd import adder
    xg = x.clone().requires_grad_(True)
    adder.adder2d_function(xg, w, 1, 0).backward(gy)
    return xg.grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matches_the_oracle(shape, dtype, gpu):
    from oracle import c_oracle
    x, w, gy = make_case(*shape, 1, 1, 0)
    x, gy = x.to(dtype), gy.to(dtype)
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, 1, 0)
    xg, wg, gyg = x.to(gpu), w.to(gpu), gy.to(gpu)
    got = _grad_x(xg, wg, gyg)
    (assert_close if dtype == torch.float32 else _close_bf16)(got, want, f"grad_x {shape}")
    off = torch.empty(gyg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(gyg).copy_(gyg)   # aligned to one element only
    assert torch.equal(_grad_x(xg, wg, off), got)


# (links are offered for whole groups of four positions and layers of 64 and more channels on both sides)
LINKED = [(2, 64, 2, 2, 66), (40, 270, 8, 8, 129), (37, 68, 8, 8, 1027), (64, 72, 14, 14, 70), (160, 65, 20, 20, 70)]


@pytest.mark.parametrize("shape", LINKED, ids=str)
def test_link_and_second_gradient_leave_the_bits(shape, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, BnLinks, bwd_bn_slots, conv_dims
    N, Ci, H, W, Co = shape
    x, w, gy = (t.to(gpu) for t in make_case(*shape, 1, 1, 0))
    x = torch.relu(x)
    gadd, bn_x, gx, out = torch.randn_like(x), torch.randn_like(x), torch.empty_like(x), torch.empty_like(x)
    mean, rstd = torch.randn(Ci, device=gpu), torch.rand(Ci, device=gpu) + 0.5
    dims, _, _ = conv_dims(x.shape, w.shape, 1, 0)
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
