"""The weight gradient of layers large enough for the 8-bit matrix cores (csrc/grad_w_i8.hip), which take them in bfloat16 storage, at the edges
of its tiles; and what fixed-point digits can lose: values far below the largest beside them, in both storage types.

Bound of ``_check``: 2^-25 ||x_ci|| ||gy_co|| beside the float32 rounding of the result.  fp64 products and the digits of values that they hold
exactly stay far within; the plain 1x1 kernel's float32 runs have at most 64 terms, each rounded by 2^-24 of a sum that grows like the root of
its terms' squares, so that a run is off by about 2^-24 of that, and the runs' errors add like their squares."""
import ctypes

import pytest
import torch

from oracle import c_oracle
from tests import test_gpu_bn_links

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, k): every tile shape and block, images not a multiple of four, channels around multiples of 16 and 32, maps that end
# inside a tile, rows that are whole groups of four and rows that are not
CASES = [(4, 16, 136, 64, 33, 3), (5, 17, 104, 33, 47, 3), (11, 30, 160, 31, 15, 3), (6, 64, 65, 29, 40, 3), (15, 33, 67, 17, 40, 3), (17, 48, 15, 16, 144, 3),
         (54, 80, 14, 14, 32, 3), (70, 130, 16, 12, 16, 3), (45, 79, 8, 8, 110, 3), (170, 90, 7, 7, 31, 3), (200, 60, 6, 5, 68, 3), (5, 16, 500, 40, 8, 3),
         (4, 3, 9, 17, 5, 5), (5, 18, 12, 33, 20, 5), (6, 16, 21, 13, 40, 5), (9, 5, 10, 16, 16, 5), (46, 40, 8, 8, 40, 5), (101, 33, 7, 6, 31, 5),
         # single taps: tiles that end inside a plane and inside a group of four, planes smaller than a group of rows, both blocks
         (1, 64, 2, 3, 64, 1), (3, 130, 7, 7, 70, 1), (2, 65, 14, 14, 129, 1), (14, 5, 15, 15, 7, 1), (11, 100, 17, 19, 33, 1), (30000, 33, 2, 2, 40, 1),
         (120, 97, 15, 15, 31, 1), (90, 40, 40, 32, 47, 1), (130, 200, 32, 20, 32, 1), (5, 70, 1, 4, 300, 1)]


# the kernel of each case in bfloat16 storage, in the dispatch's numbers: 3x3 with up to 16 output channels 20 (tiles 32 wide), 21, 22, with more 24, 25 (both
# 16 wide) and 26; 5x5 28, 29, 30; single taps 32, up to 32 output channels 33
KERNELS = [24, 26, 20, 24, 26, 25, 25, 21, 26, 26, 26, 22, 28, 29, 29, 29, 30, 30, 32, 32, 32, 33, 32, 32, 33, 32, 33, 32]


def _kernel(case, bf16):
    from addernetcuda_amd._lib import lib, check
    N, Ci, H, W, Co, k = case
    out = ctypes.c_int()
    check(lib.adder_conv2d_grad_w_kernel(N, Ci, H, W, Co, k, k, 1, k // 2, bf16, ctypes.byref(out)), "adder_conv2d_grad_w_kernel")
    return out.value


def _grad_w(gpu, x, w, gy, eta=0.0):
    from addernetcuda_amd._lib import lib, check, ptr, stream_ptr, conv_dims, conv2d_bwd_workspace
    dims, _, _ = conv_dims(x.shape, w.shape, 1, w.shape[2] // 2)
    ws, nbytes = conv2d_bwd_workspace(dims, gpu)
    gw = torch.full(w.shape, float("nan"), device=gpu)
    name = "adder_conv2d_bwd_f32" if x.dtype == torch.float32 else "adder_conv2d_bwd_bf16"
    check(getattr(lib, name)(ptr(gy), ptr(x), ptr(w), None, ptr(gw), eta, ptr(ws), nbytes, *dims, stream_ptr(gpu)), name)
    torch.cuda.synchronize()
    return gw.cpu()


def _data(case, seed):
    N, Ci, H, W, Co, k = case
    g = torch.Generator().manual_seed(seed)
    return (torch.relu(torch.randn(N, Ci, H, W, generator=g)), torch.randn(Co, Ci, k, k, generator=g),
            torch.randn(N, Co, H, W, generator=g) * 0.1)


def _check(got, x, w, gy):
    pad = w.shape[2] // 2
    want = c_oracle.conv2d_grad_w(gy, x, w, 1, pad)
    nx, ng = x.double().pow(2).sum((0, 2, 3)).sqrt(), gy.double().pow(2).sum((0, 2, 3)).sqrt()
    total = (gy.double().sum((0, 2, 3))[:, None, None, None] * w.double()).abs()   # the term of w is rounded with the sum
    bound = 2.0 ** -23 * want.abs() + 2.0 ** -25 * (ng[:, None] * nx[None, :])[:, :, None, None] + 2.0 ** -50 * total
    err = (got.double() - want).abs()
    assert bool((err <= bound).all()), f"worst element at {(err / bound).max().item():.2f} of the bound"


@pytest.mark.parametrize("case", CASES, ids=str)
def test_parity(gpu, case):
    assert not 20 <= _kernel(case, 0) < 100   # no digits in float storage
    x, w, gy = _data(case, 1)
    got = _grad_w(gpu, x.to(gpu), w.to(gpu), gy.to(gpu))
    _check(got, x, w, gy)
    assert torch.equal(got, _grad_w(gpu, x.to(gpu), w.to(gpu), gy.to(gpu)))


@pytest.mark.parametrize("case,kernel", list(zip(CASES, KERNELS)), ids=str)
def test_bfloat16_storage(gpu, case, kernel):
    assert _kernel(case, 1) == kernel
    x, w, gy = _data(case, 2)
    x, gy = x.bfloat16(), gy.bfloat16()
    _check(_grad_w(gpu, x.to(gpu), w.to(gpu), gy.to(gpu)), x.float(), w, gy.float())


@pytest.mark.parametrize("case", [CASES[0], CASES[4], CASES[9], CASES[15], CASES[19], CASES[24]], ids=str)
def test_channels_of_very_different_size_and_long_tails(gpu, case):
    x, w, gy = _data(case, 3)
    g = torch.Generator().manual_seed(4)
    x = x * torch.exp(2.0 * torch.randn(x.shape, generator=g)) * 10.0 ** (torch.rand(1, x.shape[1], 1, 1, generator=g) * 20 - 10)
    gy = gy * torch.exp(2.0 * torch.randn(gy.shape, generator=g)) * 10.0 ** (torch.rand(1, gy.shape[1], 1, 1, generator=g) * 20 - 15)
    x[:, 1] = 0.0
    gy[:, 0] = 0.0
    w = torch.zeros_like(w)   # (a sum of gy that is large against the products would hide them)
    _check(_grad_w(gpu, x.to(gpu), w.to(gpu), gy.to(gpu)), x, w, gy)


@pytest.mark.parametrize("case", [CASES[2], CASES[10], CASES[17], CASES[20], CASES[25]], ids=str)
def test_whole_numbers_are_exact(gpu, case):
    N, Ci, H, W, Co, k = case
    g = torch.Generator().manual_seed(5)
    x, w, gy = (torch.randint(-7, 8, s, generator=g).float() for s in ((N, Ci, H, W), (Co, Ci, k, k), (N, Co, H, W)))
    assert torch.equal(_grad_w(gpu, x.to(gpu), w.to(gpu), gy.to(gpu)).double(), c_oracle.conv2d_grad_w(gy, x, w, 1, k // 2).double())


@pytest.mark.parametrize("storage", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", [CASES[0], CASES[6], CASES[14], CASES[19], CASES[25], (5, 20, 21, 35, 17, 3), (3, 18, 13, 14, 20, 3), (2, 9, 7, 7, 5, 3),
                                  (6, 17, 9, 37, 18, 5), (5, 7, 6, 7, 9, 5)], ids=str)
def test_infinities_and_nan(gpu, case, storage):
    """Two infinite x and one gy that is not a number: the same elements are infinite and not a number, the others within the bound."""
    x, w, gy = _data(case, 6)
    x, gy = x.to(storage).float(), gy.to(storage).float()
    N, Ci, H, W, Co, k = case
    x[N - 1, Ci - 1, H // 2, W - 2] = float("inf")
    x[N - 1, Ci - 2, H - 1, W // 2] = float("-inf")   # (the kernels' tiles go on beside the map, where these two meet no gy)
    gy[0, 3, 1, 2] = float("nan")
    run = lambda: _grad_w(gpu, x.to(gpu, storage), w.to(gpu), gy.to(gpu, storage)).double()
    got, want = run(), c_oracle.conv2d_grad_w(gy, x, w, 1, k // 2).double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    x[N - 1, Ci - 2:] = 0.0
    gy[0, 3] = 0.0
    keep = torch.ones_like(got, dtype=torch.bool)
    keep[3], keep[:, Ci - 2:] = False, False
    clean = run()
    fine = got[keep]
    assert bool(fine.isfinite().all()) and bool(torch.isclose(fine, clean[keep], rtol=1e-6, atol=1e-5).all())


# large layers whose backward takes the BatchNorm links (float storage; the last has single taps)
@pytest.mark.parametrize("case", [(26, 20, 32, 32, 30, 1), (64, 32, 16, 16, 48, 1), (104, 64, 8, 8, 64, 1), (30, 70, 14, 14, 136, 1, 1)],
                         ids=str)
def test_linked_batchnorm(gpu, case):
    test_gpu_bn_links.test_fused_backward_matches_the_unfused_chain_in_float64(case, True, False, gpu)


@pytest.mark.parametrize("case", [(3, 18, 13, 20, 24), (2, 16, 28, 28, 17), (5, 16, 7, 4, 16)], ids=str)
def test_infinities_behind_a_linked_batchnorm(gpu, case):
    from addernetcuda_amd._lib import lib, check, ptr, stream_ptr, conv_dims, conv2d_bwd_workspace, BnLinks
    x, w, dz = _data((*case, 3), 16)
    N, Ci, H, W, Co = case
    x[N - 1, Ci - 1, H // 2, W - 1] = float("inf")
    x[N - 1, Ci - 2, H - 1, W // 2] = float("-inf")
    g = torch.Generator().manual_seed(17)
    y, coef = torch.randn(dz.shape, generator=g).to(gpu), (torch.rand(Co, 4, generator=g) * 0.1).to(gpu)
    xg, wg, dzg = x.to(gpu), w.to(gpu), dz.to(gpu)
    gx, gw, gy = torch.empty_like(xg), torch.empty_like(wg), torch.full_like(dzg, float("nan"))
    dims, _, _ = conv_dims(x.shape, w.shape, 1, 1)
    ws, nbytes = conv2d_bwd_workspace(dims, gpu)
    links = BnLinks(out_x=ptr(y), out_coef=ptr(coef), out_gy=ptr(gy))
    check(lib.adder_conv2d_bwd_bn_f32(ptr(dzg), ptr(xg), ptr(wg), None, ptr(gx), ptr(gw), 0.0, ptr(ws), nbytes, *dims, ctypes.byref(links),
                                      stream_ptr(gpu)), "adder_conv2d_bwd_bn_f32")
    torch.cuda.synchronize()
    gy, got = gy.cpu(), gw.cpu().double()
    assert bool(gy.isfinite().all())
    want = c_oracle.conv2d_grad_w(gy, x, w, 1, 1).double()
    assert bool(got.isinf().any()) and torch.equal(got.isnan(), want.isnan()) and torch.equal(got[got.isinf()], want[want.isinf()])
    fine = want.isfinite()
    assert bool(torch.isclose(got[fine], want[fine], rtol=1e-6, atol=1e-5).all())


# the entry point without a workspace, where the slabs of the bfloat16 kernels or, the last two, of the fp64 ones would not fit its scratch
@pytest.mark.parametrize("case", [(256, 32, 16, 16, 32, 3), (32, 128, 14, 14, 120, 3), (8, 48, 28, 28, 48, 5), (200, 63, 16, 16, 4096, 1),
                                  (64, 256, 14, 14, 256, 1), (40, 130, 9, 9, 1000, 1)], ids=str)
def test_without_a_workspace(gpu, case):
    from addernetcuda_amd._lib import lib, check, ptr, stream_ptr, conv_dims, conv2d_bwd_workspace
    assert _kernel(case, 1) >= 20
    x, w, gy = _data(case, 7)
    dims, _, _ = conv_dims(x.shape, w.shape, 1, case[5] // 2)
    assert conv2d_bwd_workspace(dims, gpu)[1] > 8 << 20
    xg, wg, gyg, gw = x.to(gpu), w.to(gpu), gy.to(gpu), torch.full(w.shape, float("nan"), device=gpu)
    check(lib.adder_conv2d_bwd_noalloc_f32(ptr(gyg), ptr(xg), ptr(wg), None, ptr(gw), 0.0, *dims, stream_ptr(gpu)), "noalloc")
    torch.cuda.synchronize()
    _check(gw.cpu(), x, w, gy)


@pytest.mark.parametrize("storage", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", [CASES[20], CASES[25], (9, 130, 12, 12, 140, 1), (3, 64, 4, 4, 65, 1)], ids=str)
def test_bases_between_the_groups(gpu, case, storage):
    """Tensors that begin one element into an allocation: the same results, element by element; the staged call, too."""
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims, conv2d_bwd_workspace, GradWStage
    x, w, gy = _data(case, 8)
    x, gy = x.to(storage), gy.to(storage)
    off = lambda t: torch.cat([t.new_zeros(1), t.flatten()]).to(gpu)[1:].view(t.shape)
    xo, wg, gyo = off(x), w.to(gpu), off(gy)
    assert torch.equal(_grad_w(gpu, xo, wg, gyo), _grad_w(gpu, x.to(gpu), wg, gy.to(gpu)))
    if storage == torch.float32 and min(case[1], case[4]) >= 64:
        dims, _, _ = conv_dims(x.shape, w.shape, 1, 0)
        ws, nbytes = conv2d_bwd_workspace(dims, gpu)
        gw, stage = torch.empty_like(wg), GradWStage()
        assert lib.adder_conv2d_grad_w_staged_f32(ptr(gyo), ptr(xo), ptr(wg), ptr(gw), 0.0, ptr(ws), nbytes, *dims, ctypes.byref(stage), stream_ptr(gpu)) == 0
        torch.cuda.synchronize()


# column matrices with long sums (Co, K, NL)
@pytest.mark.parametrize("case", [(17, 33, 300004), (64, 576, 12100), (130, 100, 30000)], ids=str)
def test_column_matrices(gpu, case):
    from addernetcuda_amd import adder_cuda
    Co, K, NL = case
    assert -(-Co // 16) * -(-K // 16) * 256 * NL >= 2.2e8
    x, w, gy = _data((1, K, 1, NL, Co, 1), 9)
    X, G, Wm = x.view(K, NL).to(gpu), gy.view(Co, NL).to(gpu), w.view(Co, K).to(gpu)
    gw = torch.full_like(Wm, 2.0)
    adder_cuda.ADDER_CONV_WEIGHT(G, X, Wm, gw)
    torch.cuda.synchronize()
    want = c_oracle.col_grad_w(gy.view(Co, NL), x.view(K, NL), w.view(Co, K))
    bound = 2.0 ** -23 * (want.abs() + 2.0) + 2.0 ** -25 * gy.view(Co, NL).double().norm(dim=1)[:, None] * x.view(K, NL).double().norm(dim=1)[None]
    bound += 2.0 ** -50 * (gy.double().sum((0, 2, 3))[:, None] * w.view(Co, K).double()).abs()
    assert bool(((gw.cpu().double() - 2.0 - want).abs() <= bound).all())


def _check_each(run, x, w, gy, storage, smallest=0.0):
    """Exact products and sums in fp64, element by element: the rounding of the result and 2^-45 of the sum of magnitudes.  bfloat16 storage, whose
    kernels hold the deviation of the digits' error to 2^-24 of the root mean square of a block's rows and columns: six times that of
    the largest of a row and of a column.  ``smallest``: the rounding of results below the normal floats."""
    x, gy = x.to(storage).float(), gy.to(storage).float()
    k = w.shape[2]
    got, want = run(x.to(storage), w, gy.to(storage)), c_oracle.conv2d_grad_w(gy, x, w, 1, k // 2)
    if storage == torch.bfloat16:
        smallest = smallest + 6 * 2.0 ** -24 * torch.minimum(want.abs().amax((1, 2, 3), keepdim=True), want.abs().amax((0, 2, 3), keepdim=True))
    sums = c_oracle.conv2d_grad_w(gy.abs(), x.abs(), torch.zeros(want.shape), 1, k // 2)
    bound = 2.0 ** -24 * want.abs() + 2.0 ** -45 * sums + smallest
    err = (got.double() - want).abs()
    assert bool((err <= bound).all()), f"worst element at {(err / bound).max().item():.2f} of the bound"


def _spots(t, step):
    """every step-th row and column of every image, a few of 256 neighbouring positions"""
    spots = torch.zeros(t.shape[0], 1, *t.shape[2:], dtype=torch.bool)
    spots[:, :, step // 2::step, step // 2::step] = True
    return spots


def _around(spots, k):
    return torch.nn.functional.max_pool2d(spots.float(), k, 1, k // 2) > 0


def _large_opposite_zeros(case, which, size):
    """``which`` holds large values whose partners under every tap are zeros: they contribute nothing."""
    x, w, gy = _data(case, 10)
    k = case[5]
    spots = _spots(x, 4 if k == 1 else 7)
    if which != "gy":
        x = torch.where(spots, torch.tensor(size), x)
        gy = gy.masked_fill(_around(spots, k), 0.0)
    if which != "x":
        other = spots.roll((2, 2), (2, 3)) & ~_around(spots, k) if which == "both" else spots
        gy = torch.where(other, torch.tensor(size), gy)
        x = x.masked_fill(_around(other, k), 0.0)
    return x, torch.zeros_like(w), gy   # (no w: the sum of a gy that is large is large itself)


def _run(gpu):
    return lambda x, w, gy: _grad_w(gpu, x.to(gpu), w.to(gpu), gy.to(gpu))


# tiles of 16 x 4, 8 x 8 and 32 x 2, 5x5, both blocks of single taps; float32 storage: wide enough for fp64 products (the others' are float32)
WIDE = [CASES[3], CASES[8], CASES[13], CASES[16], CASES[20]]
STORED = [(c, torch.float32) for c in WIDE] + [(c, torch.bfloat16) for c in (*WIDE, CASES[2], CASES[25])]
stored = pytest.mark.parametrize("case,storage", STORED, ids=str)


@pytest.mark.parametrize("size", [1e5, 1e30])
@pytest.mark.parametrize("which", ["x", "gy", "both"])
@stored
def test_large_values_opposite_zeros(gpu, case, storage, which, size):
    _check_each(_run(gpu), *_large_opposite_zeros(case, which, size), storage)


@pytest.mark.parametrize("share", [0.1, 0.001])
@stored
def test_sparse_gradients(gpu, case, storage, share):
    x, w, gy = _data(case, 11)
    gy = gy * (torch.rand(gy.shape, generator=torch.Generator().manual_seed(12)) < share)
    _check_each(_run(gpu), x, torch.zeros_like(w), gy, storage)


# products that are ordinary numbers of factors that are not: gradients near the smallest float and below the normal ones
@pytest.mark.parametrize("up,down", [(1.0, 1e-34), (1e10, 1e-39), (1e38, 1e-38)])
@stored
def test_tiny_and_huge_factors(gpu, case, storage, up, down):
    x, w, gy = _data(case, 13)
    _check_each(_run(gpu), x.clamp(max=3.0) * up, torch.zeros_like(w), gy * down, storage, 2.0 ** -149)


# both factors log-normal of a wide spread, and the sum of gy, which w multiplies, small against its terms
@stored
def test_long_tails(gpu, case, storage):
    x, w, gy = _data(case, 14)
    g = torch.Generator().manual_seed(15)
    x, gy = x * torch.exp(4.0 * torch.randn(x.shape, generator=g)), gy * torch.exp(4.0 * torch.randn(gy.shape, generator=g))
    _check_each(_run(gpu), x, torch.zeros_like(w), gy, storage)
    x, gy = torch.zeros_like(x), gy.to(storage).float()
    want = c_oracle.conv2d_grad_w(gy, x, w, 1, case[5] // 2)
    sums = gy.double().abs().sum((0, 2, 3))[:, None, None, None] * w.double().abs()
    got = _grad_w(gpu, x.to(gpu, storage), w.to(gpu), gy.to(gpu, storage)).double()
    assert bool(((got - want).abs() <= 2.0 ** -24 * want.abs() + 2.0 ** -45 * sums).all())


def test_column_matrix_with_large_values_opposite_zeros(gpu):
    from addernetcuda_amd import adder_cuda
    Co, K, NL = 64, 576, 12100
    x, w, gy = _large_opposite_zeros((1, K, 1, NL, Co, 1), "x", 1e9)
    x[:, :, :, ::16], gy[:, :, :, ::16] = 1e9, 0.0

    def run(x, w, gy):
        gw = torch.zeros(Co, K, device=gpu)
        adder_cuda.ADDER_CONV_WEIGHT(gy.view(Co, NL).to(gpu), x.view(K, NL).to(gpu), w.view(Co, K).to(gpu), gw)
        torch.cuda.synchronize()
        return gw.cpu().view(Co, K, 1, 1)
    _check_each(run, x, w, gy, torch.float32)
