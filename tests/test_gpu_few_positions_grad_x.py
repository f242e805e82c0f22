"""The input-gradient kernel for few positions: against the float64 oracle at its edges -- tails in positions, input channels
(the shifted last group of four) and chunks of output channels, more chunks than waves, one tap and nine, both storage
types, a second gradient added -- and against the same images in a large batch, which most shapes run on the tiled kernel."""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, k, stride, pad)
SHAPES = [(1, 4, 32, 31, 16, 3, 1, 1), (1, 64, 8, 8, 64, 3, 1, 1), (1, 64, 9, 7, 64, 3, 1, 1), (2, 33, 14, 14, 37, 3, 1, 1), (1, 6, 7, 7, 200, 3, 1, 1),
          (3, 5, 1, 1, 17, 3, 1, 1), (1, 7, 9, 33, 40, 3, 1, 1), (7, 37, 27, 19, 51, 3, 1, 1), (1, 65, 9, 7, 48, 1, 1, 0),
          (2, 66, 7, 7, 300, 1, 1, 0), (1, 127, 3, 3, 521, 1, 1, 0), (1, 64, 13, 15, 130, 1, 1, 0), (1, 256, 27, 27, 64, 1, 1, 0)]


def _grad_x(x, w, gy, case):
    from addernetcuda_amd import adder
    xg = x.clone().requires_grad_(True)
    adder.adder2d_function(xg, w, case[6], case[7]).backward(gy)
    return xg.grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_matches_the_oracle(case, dtype, gpu):
    from oracle import c_oracle
    x, w, gy = make_case(*case)
    x, gy = x.to(dtype), gy.to(dtype)
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, case[6], case[7])
    got = _grad_x(x.to(gpu), w.to(gpu), gy.to(gpu), case)
    (assert_close if dtype == torch.float32 else _close_bf16)(got, want, f"grad_x {case}")


@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_agrees_with_a_large_batch(case, gpu):
    x, w, gy = (t.to(gpu) for t in make_case(*case))
    few = _grad_x(x, w, gy, case)
    reps = 2048 // case[0] if case[2] * case[3] < 200 else 256 // case[0]
    big = _grad_x(x.repeat(reps, 1, 1, 1), w, gy.repeat(reps, 1, 1, 1), case)
    # both sum rounded products of the same size: the parity bar of either against float64, twice
    assert torch.allclose(big[:case[0]], few, rtol=2e-5, atol=2e-4)
    assert torch.equal(_grad_x(x, w, gy, case), few)     # no race: the same bits again


@pytest.mark.parametrize("case", [SHAPES[3], SHAPES[9]], ids=str)
def test_second_gradient_is_added_once(case, gpu):
    import ctypes
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    N, Ci, H, W, Co, k, s, p = case
    x, w, gy = (t.to(gpu) for t in make_case(*case))
    gadd, gx = torch.randn_like(x), torch.empty_like(x)
    gw, need = torch.empty_like(w), ctypes.c_size_t(0)
    assert lib.adder_conv2d_bwd_workspace_bytes(N, Ci, H, W, Co, k, k, s, p, ctypes.byref(need)) == 0
    ws = torch.empty(max(need.value, 256), dtype=torch.uint8, device=gpu)
    assert lib.adder_conv2d_bwd_add_f32(ptr(gy), ptr(x), ptr(w), ptr(gadd), ptr(gx), ptr(gw), 0.0, ptr(ws), need.value,
                                        N, Ci, H, W, Co, k, k, s, p, stream_ptr(x.device)) == 0
    assert torch.equal(gx, _grad_x(x, w, gy, case) + gadd)
