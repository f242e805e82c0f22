"""The lists of tests/kernel_shapes.py against the library's answers (no GPU): each layer takes the shape it stands for, and no layer takes one that no
list has.  A line of a dispatch that moves fails here, with the layer that has to be found again."""
import random

import pytest

from tests.kernel_shapes import FORWARD, GRAD_X, STATS_APART, forward_shape, grad_x_shape
from tests.util import TAP, NINE, S2, TILED_FORWARD, fwd_kernel, grad_x_kernel, stats_apart, stats_kernel


@pytest.mark.parametrize("shape", FORWARD, ids=str)
def test_forward_layers_take_their_shape(shape):
    for waves, case in FORWARD[shape].items():
        assert forward_shape(case) == (shape, waves), case
    assert set(FORWARD[shape]) == ({1} if shape == (TAP, 1, True, None, 8, 4) else {1, 2, 4, 8})


@pytest.mark.parametrize("shape", GRAD_X, ids=str)
def test_input_gradients_take_their_shape(shape):
    for waves, case in GRAD_X[shape].items():
        assert grad_x_shape(case) == grad_x_shape(case, bf16=True) == (shape, waves), case


def _layers(n):
    r = random.Random(5)
    for _ in range(n):
        k = r.choice([1, 3, 5])
        size = lambda most: int(2 ** r.uniform(0, most))
        yield size(9), size(10), size(6), size(6), size(10), k, r.choice([1, 2, 3] if k == 1 else [1, 2]), k // 2


def test_no_layer_takes_another_shape():
    for case in _layers(20000):
        if fwd_kernel(case)[0] in (TAP, NINE):
            shape, waves = forward_shape(case)
            assert waves in FORWARD[shape], case
        for bf16 in (False, True):
            if grad_x_kernel(case, bf16)[0] in (TAP, NINE, S2):
                shape, waves = grad_x_shape(case, bf16)
                assert waves in GRAD_X[shape], case


@pytest.mark.parametrize("Co,waves", [(8, 1), (9, 1), (12, 2), (17, 2), (20, 4), (33, 4), (64, 4), (65, 8)])
@pytest.mark.parametrize("k", [3, 5])
def test_no_wave_of_a_full_strided_launch_is_mostly_idle(Co, waves, k):
    assert grad_x_shape((62, 47, 58, 57, Co, k, 2, k // 2))[1] == waves
    assert grad_x_shape((1, 47, 14, 13, Co, k, 2, k // 2))[1] == (1 if Co <= 8 else 2 if Co <= 16 else 4 if Co <= 32 else 8)   # (a small one needs all)


def test_statistics_of_few_images_are_summed_behind_the_forward():
    assert set(STATS_APART) == set(TILED_FORWARD) | {51}
    for kernel, cases in STATS_APART.items():
        for case, batch in cases:
            many = (batch,) + case[1:]
            assert stats_kernel(case) == stats_kernel(many) == kernel and stats_apart(case) and not stats_apart(many), case
