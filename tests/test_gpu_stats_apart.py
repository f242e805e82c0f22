"""Forwards with statistics: those of a few images, which tile_stats_kernel sums behind the forward without tiles, are bit for bit the slots that the
same images have in a batch whose forward in tiles sums them -- for every tile shape -- and both are near the sums in float64."""
import ctypes

import pytest
import torch

from tests.kernel_shapes import STATS_APART
from tests.util import make_case

pytestmark = pytest.mark.gpu


def with_stats(x, w, stride, pad):
    from addernetcuda_amd._lib import lib, ptr, stream_ptr, conv_dims, check
    dims, Ho, Wo = conv_dims(x.shape, w.shape, stride, pad)
    slots = ctypes.c_int()
    check(lib.adder_conv2d_fwd_stats_slots(*dims, ctypes.byref(slots)), "slots")
    y = torch.empty(x.shape[0], w.shape[0], Ho, Wo, device=x.device)
    stats = torch.full((w.shape[0], slots.value, 2), float("nan"), dtype=torch.float64, device=x.device)
    check(lib.adder_conv2d_fwd_stats_f32(ptr(x), ptr(w), ptr(y), ptr(stats), slots.value, *dims, stream_ptr(x.device)), "stats")
    return y, stats


@pytest.mark.parametrize("kernel,case,batch", [(k, *c) for k, cases in STATS_APART.items() for c in cases], ids=str)
def test_the_same_bits_as_in_tiles(kernel, case, batch, gpu):
    n, s, p = case[0], case[6], case[7]
    x, w, _ = (t.to(gpu) for t in make_case(batch, *case[1:]))
    y, stats = with_stats(x, w, s, p)
    assert stats.isfinite().all()
    for first in (0, batch - n):
        few, mine = with_stats(x[first:first + n].contiguous(), w, s, p)
        slots = mine.shape[1]
        at = first // n * slots
        assert torch.equal(few, y[first:first + n]) and torch.equal(mine, stats[:, at:at + slots])
        # a slot adds deviations from a pivot in fp32, ten additions deep
        yd, count = few.double(), few.shape[0] * few.shape[2] * few.shape[3]
        spread, top = (yd.amax() - yd.amin()).item(), yd.abs().amax().item()
        one = 12 * 2.0 ** -24 * count * spread
        assert (mine[:, :, 0].sum(1) - yd.sum((0, 2, 3))).abs().max() <= one
        assert (mine[:, :, 1].sum(1) - (yd * yd).sum((0, 2, 3))).abs().max() <= 13 * 2.0 ** -24 * count * spread ** 2 + 2 * top * one


def test_a_plane_without_whole_waves_of_rows(gpu):
    """Maps lower than the second wave of a tile: its slot has no positions and holds zeros."""
    x, w, _ = (t.to(gpu) for t in make_case(2, 16, 5, 20, 6, 3, 2, 1))
    y, stats = with_stats(x, w, 2, 1)
    assert stats.isfinite().all() and (stats[:, 1::2] == 0).all()
    assert torch.allclose(stats[:, :, 0].sum(1), y.double().sum((0, 2, 3)), rtol=1e-6)


def test_statistics_under_capture(gpu):
    """Two launches of one stream: replays give the eager statistics."""
    x, w, _ = (t.to(gpu) for t in make_case(4, 32, 16, 16, 32, 3, 1, 1))
    y, want = with_stats(x, w, 1, 1)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            yg, got = with_stats(x, w, 1, 1)
    torch.cuda.synchronize()
    for k in range(3):
        x.mul_(1.0 + k)
        y, want = with_stats(x, w, 1, 1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(yg, y)
