"""1x1 / stride-1 input gradients of few channels (csrc/grad_x_tap.hip) against the float64 oracle where its groups of four, eight and sixteen input
channels, its strips, tiles and waves end -- with bases of any alignment and both storage types; a second gradient is refused as before."""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co)
SHAPES = [(1, 4, 1, 1, 16), (3, 5, 1, 2, 17), (70, 7, 1, 3, 40), (9, 8, 5, 5, 19), (200, 9, 7, 7, 131), (40, 15, 20, 21, 33), (2, 16, 9, 9, 64), (130, 23, 14, 14, 65),
          (65, 63, 9, 10, 47), (12, 63, 31, 33, 130), (9, 70, 9, 9, 33), (4, 6, 30, 31, 300),
          (40, 70, 21, 21, 40), (160, 66, 21, 21, 35)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matches_the_oracle(shape, dtype, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    x, w, gy = make_case(*shape, 1, 1, 0)
    x, gy = x.to(dtype), gy.to(dtype)
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, 1, 0)
    for base in (0, 1):   # aligned, and aligned to one element only
        g = torch.empty(gy.numel() + 1, dtype=dtype, device=gpu)[base:base + gy.numel()].view(gy.shape).copy_(gy)
        xg = x.to(gpu).requires_grad_(True)
        adder.adder2d_function(xg, w.to(gpu), 1, 0).backward(g)
        (assert_close if dtype == torch.float32 else _close_bf16)(xg.grad, want, f"grad_x {shape}, base {base}")


def test_second_gradient_is_refused(gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims
    x, w, gy = (t.to(gpu) for t in make_case(2, 24, 8, 8, 64, 1, 1, 0))
    gx = torch.empty_like(x)
    dims, _, _ = conv_dims(x.shape, w.shape, 1, 0)
    assert lib.adder_conv2d_bwd_add_f32(ptr(gy), ptr(x), ptr(w), ptr(x.clone()), ptr(gx), None, 0.0, None, 0, *dims, stream_ptr(x.device)) == -7
