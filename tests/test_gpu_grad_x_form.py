"""Input gradients that take three instructions a term and not the two that need a doubled sum minus the sum of gy: small bfloat16 layers and
ones whose rows (1x1: planes) are no whole groups of four, narrow 1x1 layers, 5x5 layers of one input channel, 3x3 and 5x5 layers on bases
aligned to one element.  An infinite gy shows which form ran: it passes through the first and is NaN in the second (inf - inf)."""
import pytest
import torch

from tests.util import make_case

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16
# (N, Ci, H, W, Co, k), storage, elements that gy's base lies beside a group of four
CASES = [((7, 63, 28, 31, 96, 3), F32, 0), ((5, 245, 23, 22, 48, 3), F32, 0), ((109, 11, 22, 22, 58, 3), F32, 0), ((8, 64, 28, 28, 64, 3), BF16, 0),
         ((16, 64, 28, 28, 64, 3), F32, 1), ((8, 256, 14, 14, 64, 1), BF16, 0), ((16, 64, 28, 28, 40, 1), F32, 0),
         ((200, 1, 32, 32, 16, 5), F32, 0), ((32, 32, 16, 16, 32, 5), F32, 1)]


@pytest.mark.parametrize("case,dtype,offset", CASES, ids=str)
def test_an_infinite_gradient_stays_infinite(case, dtype, offset, gpu):
    from addernetcuda_amd import adder
    N, Ci, H, W, Co, k = case
    x, w, gy = make_case(*case, 1, k // 2)
    gy[N - 1, Co - 1, H // 2, W // 2] = float("inf")
    xg, wg = x.to(gpu).to(dtype).requires_grad_(True), w.to(gpu)
    base = torch.empty(gy.numel() + offset, dtype=dtype, device=gpu)[offset:].view(gy.shape)
    adder.adder2d_function(xg, wg, 1, k // 2).backward(base.copy_(gy.to(gpu)))
    gx = xg.grad.cpu()
    assert not gx.isnan().any()
    # hardtanh(w - x) is zero only where both are equal: the window around the position is infinite, nothing else is
    reach = torch.zeros(N, Ci, H, W, dtype=torch.bool)
    p = k // 2
    reach[N - 1, :, max(0, H // 2 - p):H // 2 + p + 1, max(0, W // 2 - p):W // 2 + p + 1] = True
    assert torch.equal(gx.isinf(), reach)
