"""Every compiled shape of the kernels in lanes (tests/kernel_shapes.py), both storage types: forwards bit for bit against the same subtractions in the same
order, the inference epilogue against the one in a launch of its own, input gradients against the float64 oracle -- from bases of any alignment, and with
a second gradient where the entry point adds one."""
import pytest
import torch

from tests.kernel_shapes import FORWARD, GRAD_X, OFF_GROUPS
from tests.test_gpu_bf16 import _close_bf16
from tests.test_gpu_forward_order import emulate
from tests.util import assert_close, make_case

pytestmark = pytest.mark.gpu

FORWARD_CASES = [case for waves in FORWARD.values() for case in waves.values()]
GRAD_X_CASES = [case for waves in GRAD_X.values() for case in waves.values()]


def _off(t):
    """t from a base that is aligned to one element only."""
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view_as(t).copy_(t)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", FORWARD_CASES, ids=str)
def test_forward(case, dtype, gpu):
    from addernetcuda_amd import adder
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    N, Ci, H, W, Co, k, s, p = case
    x, w, _ = make_case(*case)
    x, w = x.to(gpu).to(dtype), w.to(gpu)
    y = adder.adder2d_function(x, w, s, p)
    assert torch.equal(y, emulate(x.float(), w, s, p).to(dtype))
    assert torch.equal(adder.adder2d_function(_off(x), w, s, p), y)
    if dtype == torch.bfloat16:
        return
    gamma, beta, mean, var = (torch.rand(Co, device=gpu) + 0.5 for _ in range(4))
    fused, alone, res = torch.empty_like(y), torch.empty_like(y), torch.randn_like(y)
    st = stream_ptr(x.device)
    assert lib.adder_conv2d_fwd_bn_eval_f32(ptr(x), ptr(w), ptr(fused), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5, ptr(res), 1, *case[:6], *case[5:], st) == 0
    assert lib.adder_bn_eval_f32(ptr(y), ptr(alone), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5, ptr(res), 1, N, Co, y.shape[2] * y.shape[3], st) == 0
    assert torch.equal(fused, alone)


def _grad_x(x, w, gy, s, p):
    from addernetcuda_amd import adder
    xg = x.clone().requires_grad_(True)
    adder.adder2d_function(xg, w, s, p).backward(gy)
    return xg.grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", GRAD_X_CASES + OFF_GROUPS, ids=str)
def test_grad_x(case, dtype, gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims
    from oracle import c_oracle
    s, p = case[6:]
    x, w, gy = make_case(*case)
    x, gy = x.to(dtype), gy.to(dtype)
    close = assert_close if dtype == torch.float32 else _close_bf16
    want = c_oracle.conv2d_grad_x(gy.float(), x.float(), w, s, p)
    x, w, gy = x.to(gpu), w.to(gpu), gy.to(gpu)
    got = _grad_x(x, w, gy, s, p)
    close(got, want, f"grad_x {case}")
    close(_grad_x(x, w, _off(gy), s, p), want, f"grad_x {case}, gy aligned to one element")
    if dtype == torch.bfloat16:
        return
    gadd, out = torch.randn_like(x), torch.empty_like(x)
    dims, _, _ = conv_dims(x.shape, w.shape, s, p)
    rc = lib.adder_conv2d_bwd_add_f32(ptr(gy), ptr(x), ptr(w), ptr(gadd), ptr(out), None, 0.0, None, 0, *dims, stream_ptr(x.device))
    assert rc == -7 or (rc == 0 and torch.equal(out, got + gadd))
