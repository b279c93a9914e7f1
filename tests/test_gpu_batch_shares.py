"""The batch launch's shares of rows: every split of ragged simulations (empty
and one-row ones among them) over lanes, groups per wave and limited grids
gives each row the operator that the plain launch gives it."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss
from fields import RABI_SWEEP_HALF, RABI_SWEEP_ONE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field,spin", [(RABI_SWEEP_HALF, "HALF"), (RABI_SWEEP_ONE, "ONE")])
@pytest.mark.parametrize("lanes,items,grid", [(1, 1, 0), (1, 3, 1), (3, 2, 2), (5, 8, 0), (5, 1, 3),
                                              (64, 1, 0), (7, 16, 0), (None, None, 0)])
def test_shares_cover_every_row(field, spin, lanes, items, grid):
    q = getattr(ss.SpinQuantumNumber, spin)
    sim = ss.Simulator(field.src, q)
    rows = np.array([0, 1, 63, 0, 0, 64, 65, 2, 300, 0, 257, 1, 0])
    rng = np.random.default_rng(2)
    sweep = np.tile(field.sweep, (len(rows), 1)) * rng.uniform(0.9, 1.1, (len(rows), 1))
    psi = np.eye(q.dimension)[0]
    plan = ss.BatchPlan(sim, 0.0, (rows + 0.5) * 1e-6, 1e-7, 1e-6, psi, sweep, lanes_per_step=lanes,
                        items_per_grab=items, grid_blocks=grid)
    assert plan.total == rows.sum()
    plan.u.fill_(np.nan)
    plan.run()
    for s, n in enumerate(rows):
        a = int(plan.offsets_host[s])
        ref = sim.evaluate(0.0, (n + 0.5) * 1e-6, 1e-7, 1e-6, psi, sweep[s])
        assert ref.time.shape == (n,)
        if n:
            # ten steps of at most 0.2 rad, products in another order
            assert np.abs(plan.u[a:a + n].cpu().numpy() - ref.time_evolution).max() <= 1e-14
            assert np.abs(plan.state[a:a + n].cpu().numpy() - ref.state).max() <= 1e-12
            assert np.array_equal(plan.time[a:a + n].cpu().numpy(), ref.time)
