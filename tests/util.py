"""Seeded synthetic tensors shared by the tests (CPU float32), and which kernels layers take."""
import ctypes
import math

import torch

RTOL, ATOL = 1e-5, 1e-4  # the parity bar for forward and both gradients


def make_case(N, Ci, H, W, Co, k, stride, pad, seed=0, w_init="kaiming", x_scale=1.0):
    g = torch.Generator().manual_seed(1000 + seed)
    x = torch.randn(N, Ci, H, W, generator=g) * x_scale
    K = Ci * k * k
    if w_init == "kaiming":      # std = sqrt(2 / fan_in)
        w = torch.randn(Co, Ci, k, k, generator=g) * math.sqrt(2.0 / K)
    elif w_init == "normal":     # what adder2d itself draws (adder.py:97)
        w = torch.randn(Co, Ci, k, k, generator=g)
    else:                        # test_cuda.py:64-66 scales by 5
        w = torch.randn(Co, Ci, k, k, generator=g) * 5
    Ho = (H - k + 2 * pad) // stride + 1
    Wo = (W - k + 2 * pad) // stride + 1
    gy = torch.randn(N, Co, Ho, Wo, generator=g)
    return x, w, gy


def assert_close(actual, expected, what, rtol=RTOL, atol=ATOL):
    """allclose against a float64 truth, with a readable failure message."""
    a = actual.detach().double().cpu()
    e = expected.detach().double().cpu()
    assert a.shape == e.shape, f"{what}: shape {tuple(a.shape)} vs {tuple(e.shape)}"
    err = (a - e).abs()
    bound = atol + rtol * e.abs()
    bad = err > bound
    if bad.any():
        idx = torch.nonzero(bad)[0].tolist()
        raise AssertionError(
            f"{what}: {int(bad.sum())}/{bad.numel()} elements outside rtol={rtol} atol={atol}; "
            f"max abs err {err.max().item():.3e} (|ref| max {e.abs().max().item():.3e}); first at {idx}: "
            f"{a[tuple(idx)].item()} vs {e[tuple(idx)].item()}")


def _kernel(query, case, *more):
    from addernetcuda_amd._lib import lib, check
    N, Ci, H, W, Co, k, stride, pad = case
    kernel = ctypes.c_int(-1)
    check(getattr(lib, query)(N, Ci, H, W, Co, k, k, stride, pad, *more, ctypes.byref(kernel)), query)
    return kernel.value


GENERAL, PLAIN_1X1, TILES, TAP, NINE, S2 = range(6)


def fwd_kernel(case):
    """(kernel, output channels per lane, positions per lane, waves) of the forward the library takes for (N, Ci, H, W, Co, k, stride, pad);
    TILES: strided 1x1 layers."""
    v = _kernel("adder_conv2d_fwd_kernel", case)
    return v // 100000, v // 1000 % 100, v // 100 % 10, v % 100


def stats_kernel(case):
    """The number of the kernel that the forward with statistics takes, or whose tiles group them (stats_apart)."""
    return _kernel("adder_conv2d_fwd_stats_kernel", case) % 1000


def stats_apart(case):
    """Whether the forward with statistics is the one without tiles, and sums them behind it."""
    return _kernel("adder_conv2d_fwd_stats_kernel", case) >= 1000


def grad_x_kernel(case, bf16=False):
    """(kernel, input channels per lane, positions per lane, waves, instructions a term) of the input gradient."""
    v = _kernel("adder_conv2d_grad_x_kernel", case, int(bf16))
    return v // 1000000, v // 10000 % 100, v // 1000 % 10, v // 10 % 100, v % 10


FEW_POSITIONS = 2
# every tiled kernel of the forward with statistics, by its number, on a layer whose rows (1x1: planes) are whole groups of four and on one whose are not
TILED_FORWARD = {
    10: [(2, 3, 32, 32, 18, 3, 1, 1), (1, 5, 32, 30, 18, 3, 1, 1)],
    11: [(2, 3, 24, 24, 18, 3, 1, 1), (3, 5, 24, 27, 7, 3, 1, 1)],
    12: [(3, 3, 20, 20, 18, 3, 1, 1), (1, 3, 18, 18, 18, 3, 1, 1)],
    20: [(33, 17, 13, 16, 70, 3, 1, 1), (2, 5, 9, 9, 18, 3, 1, 1)],
    30: [(1, 17, 8, 8, 18, 3, 1, 1), (5, 16, 7, 7, 17, 3, 1, 1)],
    40: [(1, 3, 20, 24, 18, 3, 2, 1), (1, 3, 20, 20, 18, 3, 2, 1), (2, 3, 18, 18, 18, 3, 2, 1)],
    50: [(1, 17, 8, 8, 18, 3, 2, 1), (1, 17, 9, 9, 18, 3, 2, 1)],
    51: [(65, 128, 16, 16, 130, 3, 2, 1), (130, 128, 9, 9, 130, 3, 2, 1)],
    60: [(1, 64, 14, 14, 18, 1, 1, 0), (1, 64, 15, 15, 18, 1, 1, 0)],
    70: [(1, 64, 8, 8, 18, 1, 1, 0), (1, 64, 7, 7, 18, 1, 1, 0)],
    80: [(16, 72, 32, 32, 70, 1, 2, 0), (33, 64, 32, 30, 70, 1, 2, 0)],
    90: [(33, 72, 24, 24, 70, 1, 2, 0), (33, 64, 17, 33, 70, 1, 2, 0)],
    100: [(1, 68, 14, 14, 18, 1, 1, 0), (1, 68, 15, 15, 18, 1, 1, 0)],
    110: [(1, 68, 8, 8, 18, 1, 1, 0), (1, 68, 7, 7, 18, 1, 1, 0)],
    120: [(1, 68, 28, 28, 18, 1, 2, 0), (1, 68, 32, 30, 18, 1, 2, 0)],
    130: [(1, 68, 8, 8, 18, 1, 2, 0), (1, 68, 7, 7, 18, 1, 3, 0)],
}
# layers of one image, with a batch that is large enough for another kernel or shape of the plain forward, by the kernel in tiles that the batch takes with
# statistics (from 60 on, 1x1 layers, one image takes the one for few positions there)
FEW_AND_TILED = {
    10: ((1, 16, 32, 32, 40, 3, 1, 1), 16), 11: ((1, 16, 24, 24, 16, 3, 1, 1), 64), 12: ((1, 16, 17, 32, 16, 3, 1, 1), 64),
    20: ((1, 33, 14, 14, 37, 3, 1, 1), 128), 30: ((1, 200, 7, 7, 31, 3, 1, 1), 2048), 40: ((1, 32, 17, 32, 33, 3, 2, 1), 256),
    50: ((1, 33, 7, 7, 40, 3, 2, 1), 256), 51: ((1, 130, 9, 9, 16, 3, 2, 1), 1024), 60: ((1, 128, 32, 32, 16, 1, 1, 0), 8),
    70: ((1, 128, 20, 20, 40, 1, 1, 0), 8), 80: ((1, 64, 28, 28, 16, 1, 2, 0), 128), 90: ((1, 64, 9, 9, 16, 1, 2, 0), 1024),
    100: ((1, 300, 32, 32, 16, 1, 1, 0), 8), 110: ((1, 300, 7, 7, 21, 1, 1, 0), 1024), 120: ((1, 300, 32, 32, 16, 1, 2, 0), 32),
    130: ((1, 300, 7, 7, 16, 1, 2, 0), 512),
}
