"""Gradients where the backward launch changes its workgroups, and where few
and many rows share a knot."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import spinsim_amd as ss

pytestmark = pytest.mark.gpu

SRC = "__device__ void get_field(double t, const double* s, double* f) { f[2] = s[0]; }"


def _gradients(sims, rows, knots, deterministic, order=1):
    grid = np.linspace(0.0, rows * 1e-6, knots)
    sim = ss.ControlledSimulator(ss.SpinQuantumNumber.HALF, [ss.Control(a, grid, order=order) for a in "xyz"], SRC)
    rng = np.random.default_rng(rows)
    a = torch.tensor(1e4 * rng.normal(size=(sims, 3, knots)), device="cuda")

    def grad(part):
        x = a[part].clone().requires_grad_()
        psi = sim.final_state(x, 0.0, (rows + 0.5) * 1e-6, 5e-7, 1e-6, [0.6, 0.8], [[2e5]] * len(x),
                              deterministic=deterministic)
        (1 - psi[:, -1].abs() ** 2).sum().backward()
        return x.grad.cpu().numpy()

    return grad(slice(None)), np.concatenate([grad(slice(s, s + 1)) for s in range(sims)])


@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("deterministic", [False, True])
def test_workgroups_of_one_wave_and_of_four(extra, deterministic):
    # 64 rows a compute unit, and a row per simulation fewer and more; alone,
    # each simulation is below
    rows = 8 * torch.cuda.get_device_properties(0).multi_processor_count + extra
    whole, alone = _gradients(8, rows, 50, deterministic)
    # the rows' terms, and their products over `rows` steps, in another order
    assert np.abs(whole - alone).max() <= 1e-11 * np.abs(alone).max()


@pytest.mark.parametrize("rows,knots", [(1, 2), (7, 8), (8, 8), (9, 3), (100, 2), (333, 97), (500, 5), (50, 100)])
@pytest.mark.parametrize("order", [1, 3])
def test_record_sums_match_atomics(rows, knots, order):
    records, _ = _gradients(2, rows, max(knots, order), True, order=order)
    atomics, _ = _gradients(2, rows, max(knots, order), False, order=order)
    assert np.abs(records - atomics).max() <= 1e-12 * np.abs(atomics).max()
