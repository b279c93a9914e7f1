"""evaluate's states around the launch sizes at which the carries get a pass of
their own and at which the scan leaves the integrator."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import spinsim_amd as ss
from fields import RABI_SWEEP_HALF, RABI_SWEEP_ONE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field,spin", [(RABI_SWEEP_HALF, "HALF"), (RABI_SWEEP_ONE, "ONE")])
@pytest.mark.parametrize("rows,fine,lanes", [(262145, 1, 1), (524289, 2, 1), (65536, 64, 64), (65537, 64, 64),
                                             (1000003, 1, 1), (4194304, 1, 1), (4194305, 1, 1)])
def test_states_follow_the_operators(field, spin, rows, fine, lanes):
    q = getattr(ss.SpinQuantumNumber, spin)
    sim = ss.Simulator(field.src, q)
    d = q.dimension
    psi = np.full(d, d ** -0.5, np.complex128)
    # times of at most half a second: the field's own phase stays small
    dt = 1e-7
    r = sim.evaluate(0.0, (rows + 0.5) * fine * dt, dt, fine * dt, psi, field.sweep, lanes_per_step=lanes,
                     output="torch")
    u, s = r.time_evolution, r.state
    assert s.shape == (rows, d) and np.array_equal(s[0].cpu().numpy(), psi)
    step = (u[:-1] * s[:-1, None, :]).sum(-1) - s[1:]
    # prefix and carry of neighbouring rows: two chains of about 100 products,
    # whose carries share the same rounding up to the last few
    assert float(step.abs().max()) <= 3e-13
    torch.cuda.synchronize()
