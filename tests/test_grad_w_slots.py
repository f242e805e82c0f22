"""The position splits of the matrix-core weight gradient, seen through the workspace they need: a layer the entry point
without a workspace took when the split was ceil(256 / blocks) is still taken, and the split never launches a round of
workgroups for a few stragglers (264 for 37 -> 51 channels).  Host code only."""
import math

import pytest


def _workspace(case):
    from addernetcuda_amd._lib import conv_dims, lib, check
    import ctypes
    N, Ci, H, W, Co, k, s, p = case
    dims, _, _ = conv_dims((N, Ci, H, W), (Co, Ci, k, k), s, p)
    need = ctypes.c_size_t(0)
    check(lib.adder_conv2d_bwd_workspace_bytes(*dims, ctypes.byref(need)), "adder_conv2d_bwd_workspace_bytes")
    return need.value


def _slots(case):
    N, Ci, H, W, Co, k, s, p = case
    return (_workspace(case) - 128 * 1024) // (8 * (Co * Ci * k * k + Co))


@pytest.mark.parametrize("case", [(7, 37, 27, 19, 51, 3, 1, 1), (32, 192, 14, 14, 192, 3, 1, 1), (256, 16, 32, 32, 16, 3, 1, 1),
                                  (128, 512, 8, 8, 512, 3, 1, 1), (64, 160, 16, 16, 208, 3, 1, 1), (1, 64, 8, 8, 64, 3, 1, 1),
                                  (2, 48, 6, 6, 40, 3, 2, 1)], ids=str)
def test_splits_of_3x3_layers(case):
    Ci, Co = case[1], case[4]
    blocks = math.ceil(Co / 16) * math.ceil(Ci / 16)
    quotient, slots = math.ceil(256 / blocks), _slots(case)
    slab = 8 * (Co * Ci * 9 + Co)
    assert slots >= 1
    assert _workspace(case) <= max(8 << 20, 128 * 1024 + quotient * slab + 256)
    last_round = slots * blocks % 256
    assert slots == 1 or last_round == 0 or last_round >= 64 or slots * blocks < 256
