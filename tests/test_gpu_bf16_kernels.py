"""bfloat16 storage through every kernel family the float32 path has (the tiled 1x1 kernels by plane size, stride and
channel count, the plain 1x1 kernels, the 3x3 tiles of 8 and 4 rows), at their edges; the bar is test_gpu_bf16.py's."""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, k, stride, pad)
SHAPES = [(2, 64, 12, 16, 48, 1, 1, 0), (5, 64, 8, 8, 72, 1, 1, 0), (2, 128, 14, 14, 136, 1, 1, 0),   # planes > 64, <= 64, 52-wide tiles
          (3, 68, 9, 9, 64, 1, 1, 0), (5, 128, 7, 7, 128, 1, 1, 0),            # planes that are not whole groups of four
          (2, 128, 28, 28, 128, 1, 2, 0), (2, 68, 18, 18, 64, 1, 2, 0), (3, 72, 10, 10, 64, 1, 2, 0),    # sampled planes
          (2, 24, 12, 12, 20, 1, 2, 0), (2, 24, 13, 11, 20, 1, 2, 0), (2, 24, 9, 7, 20, 1, 1, 0), (1, 3, 8, 8, 5, 1, 1, 0),
          (3, 16, 24, 28, 20, 3, 1, 1), (3, 16, 28, 20, 20, 3, 1, 1)]          # tiles of 8 rows, of 4 rows of two images


def _check(case, gpu, offset):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    s, p = case[6], case[7]
    x, w, gy = make_case(*case)
    xb, gb = x.bfloat16(), gy.bfloat16()
    # offset: bases that are not aligned to a group of four elements
    dev = lambda t: torch.cat([torch.zeros(offset, dtype=t.dtype), t.reshape(-1)]).to(gpu)[offset:].view(t.shape)
    xg, wg = dev(xb).requires_grad_(True), w.to(gpu).requires_grad_(True)
    y = adder.adder2d_function(xg, wg, s, p, eta=0.0)
    y.backward(dev(gb))
    torch.cuda.synchronize()
    xr, gr = xb.float(), gb.float()
    _close_bf16(y, c_oracle.conv2d_fwd(xr, w, s, p), f"forward {case}")
    _close_bf16(xg.grad, c_oracle.conv2d_grad_x(gr, xr, w, s, p), f"grad_X {case}")
    assert_close(wg.grad, c_oracle.conv2d_grad_w(gr, xr, w, s, p), f"grad_W {case}")


@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_bfloat16_kernels_match_the_oracle(case, gpu):
    _check(case, gpu, 0)


@pytest.mark.parametrize("case", [SHAPES[0], SHAPES[5], SHAPES[8], SHAPES[12]], ids=str)
def test_bfloat16_tensors_at_odd_addresses(case, gpu):
    _check(case, gpu, 1)


# plain 1x1 layers (fewer than 64 channels on a side): one slab and long sums, one slab of few positions, several slabs,
# rows that are not whole groups of four, stride 2
@pytest.mark.parametrize("case", [(256, 63, 28, 28, 1024, 1, 1, 0), (1, 9, 8, 8, 5, 1, 1, 0), (8, 63, 56, 56, 40, 1, 1, 0),
                                  (40, 24, 57, 55, 20, 1, 1, 0), (40, 24, 64, 64, 20, 1, 2, 0), (90, 17, 57, 55, 70, 1, 2, 0)], ids=str)
def test_plain_1x1_weight_gradient_is_summed_in_float64(case, gpu):
    from addernetcuda_amd import adder
    N, Ci, H, W, Co, k, s, p = case
    g = torch.Generator(device=gpu).manual_seed(8)
    x = torch.relu(torch.randn(N, Ci, H, W, device=gpu, generator=g)).bfloat16()
    w = torch.randn(Co, Ci, 1, 1, device=gpu, generator=g).requires_grad_(True)
    y = adder.adder2d_function(x, w, s, p, eta=0.0)
    gy = torch.randn(y.shape, device=gpu, generator=g).bfloat16()
    y.backward(gy)
    xs = x[:, :, ::s, ::s].double().transpose(0, 1).reshape(Ci, -1)
    gs = gy.double().transpose(0, 1).reshape(Co, -1)
    want = gs @ xs.t().contiguous() - w.detach().double().view(Co, Ci) * gs.sum(1, keepdim=True)
    # The product of two bfloat16 values has 16 bits, so fp32 sums of 64 of them hardly round; with fp64 from there on the
    # result's own rounding is left, 0.4 * 2^-24 = 2.4e-8 (fp32 to the end: 5.6e-8 to 1.2e-7, and more the longer the sums)
    assert (w.grad.double().view(Co, Ci) - want).norm() <= 5e-8 * want.norm()
    # and the finished gradient is scaled in place (adder.py:78): three more roundings
    raw, w.grad = w.grad, None
    adder.adder2d_function(x, w, s, p, eta=0.2).backward(gy)
    scaled = raw.double() / raw.double().norm() * 0.2 * raw.numel() ** 0.5
    assert (w.grad.double() - scaled).norm() <= 1e-7 * scaled.norm()
