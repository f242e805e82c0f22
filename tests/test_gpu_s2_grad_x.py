"""The input-gradient kernel of strided 3x3 and 5x5 layers (csrc/grad_x_s2.hip) against the float64 oracle where its blocks, tiles, groups of
channels and waves end: odd maps, whose last blocks are cut, maps of one row or column, input channels that do not fill a group,
output channels that end inside a chunk or give a wave none, one to eight waves -- with bases of any alignment and both storage
types; and a second gradient where the entry point adds one.  (All with two channels per lane: test_gpu_kernel_shapes has the layers of four, in both forms.)"""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co)
SHAPES = [(1, 2, 1, 1, 1), (3, 5, 1, 2, 7), (70, 9, 2, 3, 8), (2, 7, 5, 4, 9), (1, 3, 9, 9, 17), (9, 65, 7, 7, 129), (2, 6, 13, 18, 40),
          (150, 41, 17, 21, 5), (70, 70, 17, 13, 16), (20, 67, 21, 19, 32), (20, 67, 21, 22, 32), (9, 67, 21, 20, 40), (9, 64, 22, 22, 136),
          (9, 64, 21, 22, 300)]


def _grad_x(x, w, gy):
    from addernetcuda_amd import adder
    xg = x.clone().requires_grad_(True)
    adder.adder2d_function(xg, w, 2, w.shape[2] // 2).backward(gy)
    return xg.grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("k", [3, 5])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_matches_the_oracle(shape, k, dtype, gpu):
    from oracle import c_oracle
    x, w, gy = make_case(*shape, k, 2, k // 2)
    x, gy = x.to(dtype), gy.to(dtype)
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, 2, k // 2)
    xg, wg, gyg = x.to(gpu), w.to(gpu), gy.to(gpu)
    got = _grad_x(xg, wg, gyg)
    (assert_close if dtype == torch.float32 else _close_bf16)(got, want, f"grad_x {shape}")
    off = torch.empty(gyg.numel() + 1, dtype=dtype, device=gpu)[1:].view_as(gyg).copy_(gyg)   # aligned to one element only
    again = _grad_x(xg, wg, off)
    if shape[3] % 8:   # (rows of whole groups have tiles for aligned bases)
        assert torch.equal(again, got)
    (assert_close if dtype == torch.float32 else _close_bf16)(again, want, f"grad_x {shape}, gy aligned to one element")


@pytest.mark.parametrize("shape", [(2, 7, 5, 4, 9), (20, 67, 21, 22, 32), (9, 64, 22, 22, 136), (2, 3, 6, 6, 4), (2, 8, 7, 7, 4)], ids=str)
def test_second_gradient(shape, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims
    x, w, gy = (t.to(gpu) for t in make_case(*shape, 3, 2, 1))
    gadd, gx, out = torch.randn_like(x), torch.empty_like(x), torch.empty_like(x)
    dims, _, _ = conv_dims(x.shape, w.shape, 2, 1)
    st = stream_ptr(x.device)
    assert lib.adder_conv2d_bwd_f32(ptr(gy), ptr(x), ptr(w), ptr(gx), None, 0.0, None, 0, *dims, st) == 0
    rc = lib.adder_conv2d_bwd_add_f32(ptr(gy), ptr(x), ptr(w), ptr(gadd), ptr(out), None, 0.0, None, 0, *dims, st)
    if shape[1] >= 4 and shape[3] % 2 == 0:
        assert rc == 0 and torch.equal(out, gx + gadd)
    else:
        assert rc == -7   # odd rows and fewer than four channels never had one
