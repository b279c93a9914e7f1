"""evaluate's states where the integrator forms the scan's products itself:
row counts around whole waves, workgroups and the launch's limit, lanes that do
not divide a wave, against the operators it returns."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss
from fields import RABI_SWEEP_HALF, RABI_SWEEP_ONE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field,spin", [(RABI_SWEEP_HALF, "HALF"), (RABI_SWEEP_ONE, "ONE")])
@pytest.mark.parametrize("rows,fine,lanes", [
    (1, 1, None), (2, 3, 1), (63, 1, 1), (64, 1, 1), (65, 1, 1), (255, 1, 1), (256, 1, 1), (257, 1, 1),
    (21, 5, 3), (84, 5, 3), (85, 5, 3), (1000, 7, 5), (1000, 64, 33), (900, 64, 64), (16384, 2, 1),
    (16385, 2, 1), (65537, 1, 1), (262143, 1, 1), (262144, 1, 1), (262145, 1, 1), (4096, 64, 64),
    (4097, 64, 64), (21504, 3, 3), (21505, 3, 3), (5000, 10, -3)])
def test_states_follow_the_operators(field, spin, rows, fine, lanes):
    q = getattr(ss.SpinQuantumNumber, spin)
    sim = ss.Simulator(field.src, q)
    d = q.dimension
    rng = np.random.default_rng(rows)
    psi = rng.normal(size=d) + 1j * rng.normal(size=d)
    psi /= np.linalg.norm(psi)
    r = sim.evaluate(0.0, (rows + 0.5) * fine * 1e-7, 1e-7, fine * 1e-7, psi, field.sweep, lanes_per_step=lanes)
    u, s, spin_out = r.time_evolution, r.state, r.spin
    assert s.shape == (rows, d) and np.array_equal(s[0], psi)
    # about 60 products in a row, each within a few ulp of its unit columns
    assert rows == 1 or np.abs(np.einsum("nij,nj->ni", u[:-1], s[:-1]) - s[1:]).max() <= 1.5e-13
    z = (abs(s[:, 0]) ** 2 - abs(s[:, -1]) ** 2) * (0.5 if d == 2 else 1.0)
    assert np.abs(spin_out[:, 2] - z).max() <= 1e-14
    other = sim.evaluate(0.0, (rows + 0.5) * fine * 1e-7, 1e-7, fine * 1e-7, psi, field.sweep, lanes_per_step=-3)
    # the phased launch and its separate scan: rounding of `rows` operators apart
    assert np.abs(other.state - s).max() <= 1e-13 + 2e-15 * rows
