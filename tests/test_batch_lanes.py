"""Lanes per step of a batch plan outside 1..64: the launch refuses them."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss
from fields import RABI_SWEEP_HALF
from spinsim_amd import _native
from spinsim_amd.batch import default_batch_items


@pytest.mark.parametrize("lanes", [1, 63, 64, 65, 128, 10 ** 6])
@pytest.mark.parametrize("rows", [0, 1, 1000, 10 ** 9])
def test_groups_per_wave(rows, lanes):
    assert 1 <= default_batch_items(rows, lanes) <= 8


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [65, 128])
def test_launch_refuses(lanes):
    sim = ss.Simulator(RABI_SWEEP_HALF.src, ss.SpinQuantumNumber.HALF)
    sweep = np.tile(RABI_SWEEP_HALF.sweep, (3, 1))
    for given in ({"lanes_per_step": lanes}, {}):
        sim.lanes_per_step = lanes if not given else None
        plan = ss.BatchPlan(sim, 0.0, 100.5e-6, 1e-7, 1e-6, [1, 0], sweep, **given)
        with pytest.raises(_native.NativeError, match="lanes_per_step must be <= 64"):
            plan.run()
