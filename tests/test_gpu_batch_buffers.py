"""The device arrays of a batch plan are its own, each apart from the others: a
program may write any of them between runs."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import spinsim_amd as ss
from fields import RABI_SWEEP_HALF

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sims", [1, 3, 40])
def test_arrays_do_not_overlap(sims):
    sim = ss.Simulator(RABI_SWEEP_HALF.src, ss.SpinQuantumNumber.HALF)
    plan = ss.BatchPlan(sim, 0.0, 100.5e-6, 1e-7, 1e-6, [1, 0], np.tile(RABI_SWEEP_HALF.sweep, (sims, 1)),
                        with_spin=True)
    arrays = [plan.sweep, plan.offsets, plan.t0, plan.dt, plan.dt_out, plan.n_fine, plan.psi0, plan.counter,
              plan.time, plan.u, plan.state, plan.spin_out, plan.scan_ws]
    spans = sorted((a.data_ptr(), a.data_ptr() + a.numel() * a.element_size()) for a in arrays)
    assert all(end <= start for (_, end), (start, _) in zip(spans, spans[1:]))


def test_counter_may_be_cleared():
    sim = ss.Simulator(RABI_SWEEP_HALF.src, ss.SpinQuantumNumber.HALF)
    plan = ss.BatchPlan(sim, 0.0, 100.5e-6, 1e-7, 1e-6, [1, 0], np.tile(RABI_SWEEP_HALF.sweep, (3, 1))).run()
    before = plan.state.clone()
    assert plan.counter.shape == (1,) and plan.counter.dtype == torch.int64
    plan.counter.zero_()
    assert plan.offsets.cpu().tolist() == plan.offsets_host.tolist()
    plan.state.zero_()
    assert torch.equal(plan.run().state, before)
