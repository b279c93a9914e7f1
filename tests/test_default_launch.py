"""The launch that lanes_per_step = 0 stands for, by how a module computes its
step operators and how many of its workgroups a CU holds."""
from __future__ import annotations

import pytest

from spinsim_amd import _native

DIRECT, FLOAT32 = 1, 2


def launch(dim, steps, rows, fine, resident=3, phased=3):
    return _native.lib().ss_default_launch(dim, steps, rows, fine, 256, resident, phased)


@pytest.mark.parametrize("rows", [1, 1000, 65536, 138836, 10 ** 6])
@pytest.mark.parametrize("fine", [2, 7, 100])
def test_float32_waves_all_fit(rows, fine):
    for phased in (1, 2, 3, 4):
        assert launch(2, FLOAT32, rows, fine, phased=phased) == -min(3, phased)
        assert launch(3, FLOAT32, rows, fine, phased=phased) == -min(2, phased)


@pytest.mark.parametrize("dim", [2, 3])
def test_float32_rows_of_one_step_fill_the_device(dim):
    for phased in (1, 2, 4):
        assert launch(dim, FLOAT32, 4 * 10 ** 6, 1, phased=phased) == -phased


@pytest.mark.parametrize("rows", [1, 1000, 65536, 138836, 10 ** 6])
@pytest.mark.parametrize("fine", [0, 1, 7, 100])
def test_direct_takes_the_cost_model(rows, fine):
    for resident in (1, 2, 4):
        for dim in (2, 3):
            assert launch(dim, DIRECT, rows, fine, resident=resident) == \
                _native.lib().ss_default_lanes(rows, fine, 256, resident)


def test_invalid_arguments_give_one():
    for bad in ((4, DIRECT, 10, 5, 256, 3, 3), (2, DIRECT, 0, 5, 256, 3, 3), (2, FLOAT32, 10, -1, 256, 3, 3),
                (2, FLOAT32, 10, 5, 0, 3, 3), (2, FLOAT32, 10, 5, 256, 0, 3), (2, FLOAT32, 10, 5, 256, 3, 0)):
        assert _native.lib().ss_default_launch(*bad) == 1
