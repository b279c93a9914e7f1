"""The default launch's lanes per coarse step: within what the kernels take,
one lane where rows fill the device, more where they do not."""
from __future__ import annotations

import pytest

from spinsim_amd import _native


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 5000, 10 ** 5, 10 ** 7, 1 << 40])
@pytest.mark.parametrize("fine", [0, 1, 2, 10, 63, 64, 65, 1000, 2 ** 31 - 1])
def test_default_lanes_range(rows, fine):
    g = _native.lib().ss_default_lanes(rows, fine, 256, 3)
    assert 1 <= g <= min(64, max(1, fine))
    if rows >= 10 ** 7:
        assert g == 1
    if rows <= 64 and 2 <= fine <= 64:
        assert g == fine


def test_invalid_arguments_give_one():
    lib = _native.lib()
    for args in ((0, 5, 256, 3), (10, -1, 256, 3), (10, 5, 0, 3), (10, 5, 256, 0)):
        assert lib.ss_default_lanes(*args) == 1
