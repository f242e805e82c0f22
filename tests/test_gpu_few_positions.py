"""Forwards of few positions (small batches and maps; one position per lane, and with statistics of 1x1 layers a kernel of their own): against
the float64 oracle at their edges -- maps of 1 to 32, tails in positions, channels and channel chunks, strides, more chunks than waves -- with
statistics and both storage types; and the same bits as in a batch large enough for another kernel or shape."""
import pytest
import torch

from tests.util import make_case, assert_close, fwd_kernel, stats_kernel, FEW_AND_TILED, FEW_POSITIONS
from tests.test_gpu_bf16 import _close_bf16

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, k, stride, pad)
SHAPES = [(1, 16, 32, 32, 16, 3, 1, 1), (1, 64, 8, 8, 64, 3, 1, 1), (2, 33, 14, 14, 37, 3, 1, 1), (1, 200, 7, 7, 31, 3, 1, 1),
          (3, 33, 1, 1, 5, 3, 1, 1), (1, 40, 9, 33, 6, 3, 1, 1), (1, 32, 17, 32, 33, 3, 2, 1), (2, 130, 15, 7, 18, 3, 2, 1),
          (1, 200, 8, 8, 48, 1, 1, 0), (2, 300, 7, 7, 21, 1, 1, 0), (1, 132, 14, 14, 64, 1, 2, 0), (1, 512, 4, 4, 40, 1, 3, 0)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_few_positions_match_the_oracle(case, dtype, gpu):
    from addernetcuda_amd import adder
    from oracle import c_oracle
    assert fwd_kernel(case)[2] == 1 and (case[5] == 3 or stats_kernel(case) == FEW_POSITIONS)
    s, p = case[6], case[7]
    x, w, _ = make_case(*case)
    x = x.to(dtype)
    want = c_oracle.conv2d_fwd(x.float(), w, s, p)
    y = adder.adder2d_function(x.to(gpu), w.to(gpu), s, p)
    (assert_close if dtype == torch.float32 else _close_bf16)(y, want, f"forward {case}")
    if dtype == torch.float32:
        y2, stats = adder.adder2d_function_with_stats(x.to(gpu), w.to(gpu), s, p)
        assert_close(y2, want, f"forward with statistics {case}")
        tot = stats.sum(dim=1).cpu()
        assert torch.allclose(tot[:, 0], want.sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-3)
        assert torch.allclose(tot[:, 1], (want * want).sum(dim=(0, 2, 3)), rtol=1e-5, atol=1e-2)


@pytest.mark.parametrize("kernel", FEW_AND_TILED)
def test_same_bits_as_in_a_large_batch(kernel, gpu):
    from addernetcuda_amd import adder
    case, batch = FEW_AND_TILED[kernel]
    assert fwd_kernel(case) != fwd_kernel((batch,) + case[1:]) and stats_kernel((batch,) + case[1:]) == kernel
    x, w, _ = make_case(*case)
    xg, wg = x.to(gpu), w.to(gpu)
    few = adder.adder2d_function(xg, wg, case[6], case[7])
    big = adder.adder2d_function(xg.repeat(batch, 1, 1, 1), wg, case[6], case[7])
    assert torch.equal(big, few.expand_as(big))
    for images in (1, batch):
        y, stats = adder.adder2d_function_with_stats(xg.repeat(images, 1, 1, 1), wg, case[6], case[7])
        assert stats is not None and torch.equal(y, few.expand_as(y))
