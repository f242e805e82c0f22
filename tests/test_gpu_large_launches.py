"""Launches and tensors near the 32-bit limits: narrow maps of few channels and very many images, whose workgroups outnumber 2^23, and one image of more
than 2^30 elements.  Against the same layers in small, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_forward_of_many_narrow_maps(gpu):
    from addernetcuda_amd import adder
    n = 12_000_000                       # 5 x 5 maps, 3e8 positions of five output channels: 1.5e9 elements
    w = torch.randn(5, 1, 5, 5, generator=torch.Generator().manual_seed(0)).to(gpu)
    x = torch.empty(n, 1, 5, 5, device=gpu).normal_(generator=torch.Generator(gpu).manual_seed(1))
    y = adder.adder2d_function(x, w, 1, 2)
    for part in (slice(0, 50), slice(n // 2, n // 2 + 50), slice(n - 50, n)):
        assert torch.equal(y[part], adder.adder2d_function(x[part].clone(), w, 1, 2))


def test_input_gradient_of_many_narrow_maps(gpu):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    n = 12_000_000
    w = torch.randn(1, 5, 5, 5, generator=torch.Generator().manual_seed(0)).to(gpu)
    gen = torch.Generator(gpu).manual_seed(1)
    x, gy = torch.empty(n, 5, 5, 5, device=gpu).normal_(generator=gen), torch.empty(n, 1, 5, 5, device=gpu).normal_(generator=gen)

    def grad_x(x, gy):
        gx = torch.empty_like(x)
        dims = (x.shape[0], 5, 5, 5, 1, 5, 5, 1, 2, stream_ptr(x.device))
        assert lib.adder_conv2d_bwd_f32(ptr(gy), ptr(x), ptr(w), ptr(gx), None, 0.0, None, 0, *dims) == 0
        return gx

    gx = grad_x(x, gy)
    for part in (slice(0, 50), slice(n // 2, n // 2 + 50), slice(n - 50, n)):
        assert torch.equal(gx[part], grad_x(x[part].clone(), gy[part].clone()))


def test_forward_of_one_large_image(gpu):
    from addernetcuda_amd import adder
    from tests.test_gpu_forward_order import emulate
    x = torch.empty(1, 65, 4096, 4096, device=gpu).normal_(generator=torch.Generator(gpu).manual_seed(1))
    w = torch.randn(4, 65, 3, 3, generator=torch.Generator().manual_seed(0))
    y = adder.adder2d_function(x, w.to(gpu), 1, 1)
    for at in (0, 4096 - 20):            # the corners: their other two sides are cut off again
        crop = emulate(x[:, :, at:at + 20, at:at + 20].cpu(), w, 1, 1)
        keep = slice(0, 19) if at == 0 else slice(1, 20)
        got = y[:, :, at:at + 20, at:at + 20].cpu()
        assert torch.equal(got[:, :, keep, keep], crop[:, :, keep, keep])
