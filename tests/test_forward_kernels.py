"""Which kernels the library takes for the layers that tests send to a certain one (host code only, by the functions the launches use): a dispatch
rule that moves a layer elsewhere shows here instead of leaving a kernel untested."""
import ctypes

from tests.util import (FEW_AND_TILED, FEW_POSITIONS, GENERAL, NINE, PLAIN_1X1, S2, TAP, TILED_FORWARD, TILES, fwd_kernel, grad_x_kernel,
                        stats_kernel)


def test_layers_reach_the_tiled_kernels_they_are_listed_for():
    for kernel, cases in TILED_FORWARD.items():
        assert [stats_kernel(c) for c in cases] == [kernel] * len(cases), cases
        rows = [(c[3] if c[5] > 1 else c[2] * c[3]) % 4 == 0 for c in cases]
        assert True in rows and (False in rows or kernel in (80, 90, 120, 130)), cases   # (a strided 1x1 layer samples x)


def test_layers_change_kernel_with_the_batch():
    assert set(FEW_AND_TILED) == set(TILED_FORWARD)
    for kernel, (case, batch) in FEW_AND_TILED.items():
        many = (batch,) + case[1:]
        assert fwd_kernel(case) != fwd_kernel(many), case
        assert stats_kernel(many) == kernel and stats_kernel(case) == (FEW_POSITIONS if case[5] == 1 else kernel), case


def test_layers_beyond_the_grid_of_the_few_positions_kernel_stay_tiled():
    # four output channels per workgroup, at most 65535 workgroups
    assert stats_kernel((1, 256, 1, 1, 4 * 65535, 1, 2, 0)) == FEW_POSITIONS
    assert stats_kernel((1, 256, 1, 1, 4 * 65535 + 1, 1, 2, 0)) == 90


def test_kernels_of_some_layers():
    assert fwd_kernel((32, 64, 56, 56, 64, 3, 1, 1)) == (NINE, 8, 4, 4)
    assert fwd_kernel((1, 1, 4, 4, 1, 3, 3, 1))[0] == GENERAL
    assert fwd_kernel((64, 24, 32, 32, 48, 1, 1, 0))[0] == PLAIN_1X1
    assert fwd_kernel((32, 256, 56, 56, 512, 1, 2, 0))[0] == TILES and fwd_kernel((1, 256, 56, 56, 512, 1, 2, 0))[0] == TAP
    assert grad_x_kernel((128, 128, 32, 32, 128, 3, 1, 1))[0] == TILES
    assert grad_x_kernel((32, 64, 56, 56, 64, 3, 1, 1)) == (NINE, 8, 4, 8, 2)
    assert grad_x_kernel((7, 63, 28, 31, 96, 3, 1, 1)) == (NINE, 4, 1, 8, 3)
    assert grad_x_kernel((32, 256, 14, 14, 1024, 1, 1, 0)) == (TAP, 16, 2, 8, 2)
    assert grad_x_kernel((5, 107, 23, 23, 278, 3, 2, 1))[0] == S2
    # three instructions a term: small shapes until the chip is full, whole groups of waves
    assert grad_x_kernel((1, 174, 42, 42, 921, 3, 1, 1)) == (NINE, 4, 1, 8, 3) and grad_x_kernel((128, 512, 8, 8, 512, 3, 1, 1)) == (NINE, 8, 4, 8, 3)
    assert grad_x_kernel((32, 96, 28, 28, 17, 3, 1, 1)) == (NINE, 8, 4, 2, 2) and grad_x_kernel((32, 96, 28, 28, 33, 3, 1, 1)) == (NINE, 8, 4, 4, 2)
    assert grad_x_kernel((1, 3, 8, 8, 3, 1, 1, 0))[0] == PLAIN_1X1 and grad_x_kernel((1, 3, 8, 8, 3, 1, 3, 0))[0] == GENERAL


def test_the_queries_refuse_what_the_calls_refuse():
    from addernetcuda_amd._lib import lib
    kernel = ctypes.c_int()
    for query, more in ((lib.adder_conv2d_fwd_kernel, ()), (lib.adder_conv2d_fwd_stats_kernel, ()), (lib.adder_conv2d_grad_x_kernel, (0,))):
        assert query(1, 1, 4, 4, 1, 3, 3, 1, 1, *more, None) == -1
        assert query(0, 1, 4, 4, 1, 3, 3, 1, 1, *more, ctypes.byref(kernel)) == -2
        assert query(1, 1, 4, 4, 1, 3, 3, 3, 1, *more, ctypes.byref(kernel)) == 0 and kernel.value == 0
