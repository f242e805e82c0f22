"""Which forward kernel the library takes for the layers that tests send to a certain one (host code only): a dispatch rule
that moves a layer elsewhere shows here instead of leaving a kernel untested."""
import ctypes

from tests.util import FEW_AND_TILED, FEW_POSITIONS, TILED_FORWARD, fwd_kernel


def test_layers_reach_the_tiled_kernels_they_are_listed_for():
    for kernel, cases in TILED_FORWARD.items():
        assert [fwd_kernel(c) for c in cases] == [kernel] * len(cases), cases
        rows = [(c[3] if c[5] > 1 else c[2] * c[3]) % 4 == 0 for c in cases]
        assert True in rows and (False in rows or kernel in (80, 90, 120, 130)), cases   # (a strided 1x1 layer samples x)


def test_layers_change_from_the_few_positions_to_the_tiled_kernel_with_the_batch():
    assert set(FEW_AND_TILED) == {k for k in TILED_FORWARD if k < 140}      # (5x5 layers have no kernel for few positions)
    for kernel, (case, batch) in FEW_AND_TILED.items():
        assert fwd_kernel(case) == FEW_POSITIONS and fwd_kernel((batch,) + case[1:]) == kernel, case


def test_layers_beyond_the_grid_of_the_few_positions_kernel_stay_tiled():
    # four output channels per workgroup, at most 65535 workgroups
    assert fwd_kernel((1, 256, 1, 1, 4 * 65535, 3, 1, 1)) == FEW_POSITIONS
    assert fwd_kernel((1, 256, 1, 1, 4 * 65535 + 1, 3, 1, 1)) == 30


def test_the_query_refuses_what_the_forward_refuses():
    from addernetcuda_amd._lib import lib
    kernel = ctypes.c_int()
    assert lib.adder_conv2d_fwd_kernel(1, 1, 4, 4, 1, 3, 3, 1, 1, None) == -1
    assert lib.adder_conv2d_fwd_kernel(0, 1, 4, 4, 1, 3, 3, 1, 1, ctypes.byref(kernel)) == -2
    assert lib.adder_conv2d_fwd_kernel(1, 1, 4, 4, 1, 3, 3, 3, 1, ctypes.byref(kernel)) == 0 and kernel.value == 0
    assert lib.adder_conv2d_fwd_kernel(1, 1, 4, 4, 1, 1, 1, 1, 0, ctypes.byref(kernel)) == 0 and kernel.value == 1
