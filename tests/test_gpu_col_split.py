"""Column-matrix kernels at the lines of their dispatch: forward tiles whose waves split the rows of X, input gradients of
more than 32 output channels, weight-gradient slabs that fill whole rounds of workgroups."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (Co, K, NL).  Forward: 512 workgroups of 512 columns and one fewer, even and odd NL; 512 and 128 tiles of 128 columns, and
# one fewer; rows of X that do not divide by four waves or by a block of 256; fewer rows than waves; tiles of 256 columns: 512 and 386
# of them, one row and two more, an NL that is no multiple of four.
FORWARD = [(16, 37, 512 * 512), (16, 37, 511 * 512), (16, 20, 511 * 512 + 1), (16, 20, 511 * 512 - 1), (17, 259, 256 * 128),
           (17, 259, 255 * 128), (33, 513, 255 * 64 + 1), (16, 130, 128 * 128), (16, 130, 127 * 128), (20, 257, 16 * 1024),
           (16, 3, 65536), (15, 1, 65538), (100, 2, 16386),
           (32, 37, 65540), (20, 259, 65284), (17, 3, 65282), (32, 66, 49408), (32, 66, 49152), (33, 257, 43520), (32, 512, 49664)]
# Input gradient: one output channel above 32, around the folds at 64 and the blocks of 512, rows of X around groups of
# eight, columns around 256; grad_W: 9 blocks (504 workgroups), more than 512 blocks (one slab)
BACKWARD = [(33, 8, 2049), (63, 9, 2303), (64, 7, 2304), (65, 17, 2305), (511, 8, 2052), (512, 11, 2053), (513, 8, 2052),
            (521, 3, 2049), (1030, 9, 2051), (32, 37, 65540), (17, 9, 65537), (31, 66, 65538), (32, 288, 4096), (64, 576, 4100), (260, 2304, 2064)]


def _data(Co, K, NL, gpu, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    return (torch.randn(K, NL, device=gpu, generator=g), torch.randn(Co, K, device=gpu, generator=g),
            torch.randn(Co, NL, device=gpu, generator=g))


@pytest.mark.parametrize("case", FORWARD, ids=str)
def test_forward(case, gpu):
    from addernetcuda_amd import adder_cuda
    X, W, _ = _data(*case, gpu, 3)
    X[:, -1] = float("inf")                              # a column of its own: no other sees it
    out = torch.full((case[0], case[2]), 7.0, device=gpu)
    adder_cuda.ADDER_CONV(X, W, out)
    want = torch.stack([-(w.double()[:, None] - X.double()).abs().sum(0) for w in W])
    assert torch.isinf(out[:, -1]).all() and (out[:, -1] < 0).all()
    # first-level sums of at most 64 terms, at most K / 64 + 4 of those: 2^-24 * (64 + K / 64 + 4) of the result
    bound = 2.0 ** -24 * (64 + case[1] / 64 + 4) * want[:, :-1].abs() + 1e-6
    assert ((out[:, :-1].double() - want[:, :-1]).abs() <= bound).all()


def test_forward_of_bases_between_the_groups(gpu):
    """Tensors that begin two elements into an allocation take tiles of pairs: the same sums in the same order."""
    from addernetcuda_amd import adder_cuda
    X, W, _ = _data(32, 66, 49664, gpu, 6)
    out, off = torch.empty(32, 49664, device=gpu), torch.empty(32 * 49664 + 2, device=gpu)[2:].view(32, 49664)
    adder_cuda.ADDER_CONV(X, W, out)
    adder_cuda.ADDER_CONV(torch.cat([X.new_zeros(2), X.flatten()])[2:].view(66, 49664), W, off)
    assert torch.equal(out, off)


# one matrix per forward tile: unsplit by pairs and by single columns, split 16 x 128, 16 x 64, 8 x 128 and 8 x 64
@pytest.mark.parametrize("K", [1000, 1025, 2016, 2049, 2200])
@pytest.mark.parametrize("Co,NL", [(64, 65536), (128, 32767), (16, 65536), (33, 22001), (16, 16384), (16, 8191)], ids=str)
def test_forward_of_many_rows_sums_in_two_levels(Co, NL, K, gpu):
    from addernetcuda_amd import adder_cuda
    X, W, _ = _data(Co, K, NL, gpu, 6)
    out = torch.empty(Co, NL, device=gpu)
    adder_cuda.ADDER_CONV(X, W, out)
    want = torch.stack([-(w.double()[:, None] - X.double()).abs().sum(0) for w in W])
    # The terms have one sign: a sum of n rounds to about 0.4 * 2^-24 * sqrt(n / 3) of itself.  First-level sums of
    # n1 <= 64 of which n2 are added up: sqrt((n1 / n2 + n2) / 3), at most 3.5 for 2200 rows in one wave (n2 = 35), 8.3e-8;
    # four waves that share the rows do better.  Sums of 250 terms and more, carried from block to block: from 1.1e-7.
    assert (out.double() - want).norm() <= 1e-7 * want.norm()


@pytest.mark.parametrize("case", BACKWARD, ids=str)
def test_backward(case, gpu):
    from addernetcuda_amd import adder_cuda
    Co, K, NL = case
    X, W, G = _data(*case, gpu, 4)
    gw, gx = torch.ones_like(W), torch.ones_like(X)      # accumulated into
    adder_cuda.ADDER_BACKWARD(G, X, W, gw, gx)
    Xd, Wd, Gd = X.double(), W.double(), G.double()
    want = torch.stack([((Wd[:, k, None] - Xd[k]).clamp(-1, 1) * Gd).sum(0) for k in range(K)])
    size = torch.stack([((Wd[:, k, None] - Xd[k]).clamp(-1, 1) * Gd).abs().sum(0) for k in range(K)])
    # the difference w - x and the products round once each; sums of at most 64 terms, then Co / 64 of those.  Up to 32
    # output channels the clamp is 2 sat(..) - 1: the sum of |gy| stands in for that of the products
    size = torch.maximum(size, Gd.abs().sum(0)) if Co <= 32 else size
    assert ((gx.double() - 1 - want).abs() <= 2.0 ** -24 * (64 + Co / 64 + 8) * (size + 1) * (2 if Co <= 32 else 1)).all()
    want_w = Gd @ Xd.t() - Wd * Gd.sum(1, keepdim=True)
    # fp64 products and sums, one rounding of each of the two terms and of the result
    size_w = Gd.abs() @ Xd.abs().t() + Wd.abs() * Gd.abs().sum(1, keepdim=True)
    assert ((gw.double() - 1 - want_w).abs() <= 2.0 ** -24 * 4 * (size_w + 1)).all()


@pytest.mark.parametrize("case", [(32, 288, 1024), (3, 2050, 513), (16, 144, 65544), (9, 20, 70004), (24, 50, 66000), (33, 17, 2305),
                                  (20, 100, 2051), (32, 288, 4096)], ids=str)
def test_gradients_written_instead_of_added(case, gpu):
    from addernetcuda_amd import adder_cuda
    X, W, G = _data(*case, gpu, 5)
    gw, gx = torch.zeros_like(W), torch.zeros_like(X)
    adder_cuda.ADDER_BACKWARD(G, X, W, gw, gx)
    gw2, gx2 = torch.full_like(W, float("nan")), torch.full_like(X, float("nan"))
    adder_cuda.backward_set(G, X, W, gw2, gx2)
    assert torch.equal(gw, gw2) and torch.equal(gx, gx2)
