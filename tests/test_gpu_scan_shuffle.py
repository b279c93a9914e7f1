"""The single-simulation scan where its products start to move by shuffles."""
from __future__ import annotations

import pytest

from test_gpu_scan_blocks import test_states_follow_the_operators as states_follow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("blocks,extra", [(1536, 0), (1536, 1), (1600, -3), (3000, 129)])
def test_both_sides(dim, blocks, extra):
    states_follow(dim, blocks, extra)
