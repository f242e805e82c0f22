"""5x5 / pad 2 layers: the tiled forward, input-gradient and matrix-core weight-gradient kernels at the edges of their tiles
(8, 16 and 32 positions wide, remainders in rows, images and channels) and at the least channels they take; both storage types;
the entry point without a workspace on a layer whose slabs do not fit it.  The bars are those of the other layers."""
import pytest
import torch

from tests.util import make_case, assert_close
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, k, stride, pad)
SHAPES = [(2, 16, 32, 32, 16, 5, 1, 2), (1, 5, 9, 33, 19, 5, 1, 2), (3, 2, 17, 20, 3, 5, 1, 2), (2, 1, 8, 24, 4, 5, 1, 2),
          (2, 17, 16, 16, 70, 5, 1, 2), (1, 33, 18, 9, 33, 5, 1, 2), (5, 16, 8, 8, 48, 5, 1, 2), (6, 9, 7, 7, 17, 5, 1, 2),
          (1, 3, 1, 4, 2, 5, 1, 2), (2, 20, 32, 32, 18, 5, 2, 2), (3, 17, 15, 17, 16, 5, 2, 2), (5, 16, 16, 16, 33, 5, 2, 2),
          (3, 3, 13, 7, 5, 5, 2, 2)]


def _check(case, gpu, dtype, offset=0):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    s, p = case[6], case[7]
    x, w, gy = make_case(*case)
    x, gy = x.to(dtype), gy.to(dtype)
    dev = lambda t: torch.cat([torch.zeros(offset, dtype=t.dtype), t.reshape(-1)]).to(gpu)[offset:].view(t.shape)
    xg, wg = dev(x).requires_grad_(True), w.to(gpu).requires_grad_(True)
    y = adder.adder2d_function(xg, wg, s, p, eta=0.0)
    y.backward(dev(gy))
    torch.cuda.synchronize()
    x, gy = x.float(), gy.float()
    close = assert_close if dtype == torch.float32 else _close_bf16
    close(y, c_oracle.conv2d_fwd(x, w, s, p), f"forward {case}")
    close(xg.grad, c_oracle.conv2d_grad_x(gy, x, w, s, p), f"grad_X {case}")
    assert_close(wg.grad, c_oracle.conv2d_grad_w(gy, x, w, s, p), f"grad_W {case}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_5x5_layers_match_the_oracle(case, dtype, gpu):
    _check(case, gpu, dtype)


@pytest.mark.parametrize("case", [SHAPES[0], SHAPES[4], SHAPES[9]], ids=str)
def test_5x5_tensors_at_odd_addresses(case, gpu):
    _check(case, gpu, torch.float32, offset=1)


@pytest.mark.parametrize("Ci", [272, 280, 813, 1024])
@pytest.mark.parametrize("H,stride", [(20, 1), (12, 1), (7, 1), (20, 2), (13, 2)])
def test_5x5_forward_of_many_channels_keeps_its_precision(H, stride, Ci, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    x, w, _ = make_case(1, Ci, H, H, 16, 5, stride, 2, w_init="normal")
    want = c_oracle.conv2d_fwd(x, w, stride, 2)
    got = adder.adder2d_function(x.to(gpu), w.to(gpu), stride, 2).double().cpu()
    # One-signed terms: sums of 400 of which n2 = Ci / 16 are added up round to 0.4 * 2^-24 * sqrt((400 / n2 + n2) / 3) of the result --
    # what the layer had as 16-channel sums without tiles (of 200, Ci / 8: 1.6e-7 at 813 channels against 1.1e-7)
    n2 = Ci / 16
    assert (got - want).norm() <= 1.2 * 0.4 * 2.0 ** -24 * ((400 / n2 + n2) / 3) ** 0.5 * want.norm()


@pytest.mark.parametrize("Co", [1, 2, 4, 9])
@pytest.mark.parametrize("H", [24, 16, 7])
def test_5x5_grad_x_of_few_output_channels_keeps_its_precision(H, Co, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    x, w, gy = make_case(4, 16, H, H, Co, 5, 1, 2)
    want = c_oracle.conv2d_grad_x(gy, x, w, 1, 2)
    xg = x.to(gpu).requires_grad_(True)
    adder.adder2d_function(xg, w.to(gpu), 1, 2).backward(gy.to(gpu))
    # Terms of either sign: adding n of them rounds to 0.4 * 2^-24 * sqrt(n / 2) of the result, here sums of at most 50 and Co / 2 of
    # those, and a term's difference to about one addition.  (Two-instruction form, 2 sum d g - sum g: 1.8e-7 to 2.4e-7.)
    bound = 0.4 * 2.0 ** -24 * (min(25 * Co, 50) / 2 + Co / 4 + 1) ** 0.5
    assert (xg.grad.double().cpu() - want).norm() <= 1.2 * bound * want.norm()


def test_without_a_workspace_where_the_slabs_do_not_fit(gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims, check, conv2d_bwd_workspace
    from oracle import c_oracle
    case = (1, 160, 4, 4, 272, 5, 1, 2)      # one slab of 160 * 25 * 272 doubles is more than 8 MiB
    x, w, gy = make_case(*case)
    dims, _, _ = conv_dims(x.shape, w.shape, 1, 2)
    assert conv2d_bwd_workspace(dims, gpu)[1] > 8 << 20
    xg, wg, gg = x.to(gpu), w.to(gpu), gy.to(gpu)
    gx, gw = torch.full_like(xg, float("nan")), torch.full_like(wg, float("nan"))
    check(lib.adder_conv2d_bwd_noalloc_f32(ptr(gg), ptr(xg), ptr(wg), ptr(gx), ptr(gw), 0.0, *dims, stream_ptr(gpu)),
          "adder_conv2d_bwd_noalloc_f32")
    torch.cuda.synchronize()
    assert_close(gx, c_oracle.conv2d_grad_x(gy, x, w, 1, 2), "grad_X")
    assert_close(gw, c_oracle.conv2d_grad_w(gy, x, w, 1, 2), "grad_W")
