"""Lanes per step of a batch plan outside 1..64: the launch refuses them."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss
from fields import RABI_SWEEP_HALF
from spinsim_amd import _native
from spinsim_amd.batch import default_batch_items, default_batch_lanes


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


@pytest.mark.parametrize("cus", [32, 64, 256])
@pytest.mark.parametrize("rows,fine", [(1, 10), (2000, 7), (20000, 20), (300000, 100)])
def test_default_lanes_of_the_device(rows, fine, cus):
    """The batch default follows the device's compute units."""
    lanes = _native.lib().ss_default_lanes(rows, fine, cus, 3)
    assert default_batch_lanes(rows, fine, cus=cus) == lanes
    assert default_batch_lanes(rows, fine, float32=True, cus=cus) == default_batch_lanes(rows, fine, True)


@pytest.mark.gpu
def test_plan_follows_the_device():
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    sim = ss.Simulator(RABI_SWEEP_HALF.src, ss.SpinQuantumNumber.HALF)
    plan = ss.BatchPlan(sim, 0.0, 100.5e-6, 1e-7, 1e-6, [1, 0], np.tile(RABI_SWEEP_HALF.sweep, (30, 1)))
    assert plan.lanes == default_batch_lanes(3000, 10, cus=cus)
