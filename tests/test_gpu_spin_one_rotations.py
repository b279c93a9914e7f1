"""Spin one without a quadratic shift (accumulated as spin-half operators)
against the same field with a zero the compiler cannot see (3x3 operators), over
step sizes on both sides of its ranges, lanes per row and long chunks."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss

pytestmark = pytest.mark.gpu

FIELD = """__device__ void get_field(double t, const double* s, double* f)
{ f[0] = s[0] * cos(3e6 * t); f[1] = s[0] * sin(2e6 * t + 1); f[2] = s[0] * 0.7; %s }"""


# angle per step: inside 0.018, across it, across 1/4, beyond
@pytest.mark.parametrize("angle", [1e-4, 0.012, 0.03, 0.3, 3.0])
@pytest.mark.parametrize("method", ["MAGNUS_CF4", "EULER", "HEUN"])
@pytest.mark.parametrize("frame", [True, False])
@pytest.mark.parametrize("lanes,fine", [(None, 10), (1, 1), (3, 7), (-2, 12), (1, 1023), (1, 2500)])
def test_rotation_matches_general(angle, method, frame, lanes, fine):
    dt, rows = 1e-8, 70
    sweep = [angle / dt, 0.0]
    got = []
    for q in ("", "f[3] = s[1];"):
        sim = ss.Simulator(FIELD % q, ss.SpinQuantumNumber.ONE, use_rotating_frame=frame,
                           integration_method=getattr(ss.IntegrationMethod, method))
        r = sim.evaluate(0.0, (rows + 0.5) * fine * dt, dt, fine * dt, [0.6, 0.0, 0.8j], sweep, lanes_per_step=lanes)
        got.append((r.time_evolution, r.state, r.spin))
    u = got[0][0]
    # both round each of up to 5000 factors at most a few ulp of the larger of
    # its angle and the chunk's residual (below 3)
    tol = 2e-15 + 2 * fine * 3 * 2.2e-16
    assert np.abs(u - got[1][0]).max() <= tol
    assert np.abs(np.conj(u.transpose(0, 2, 1)) @ u - np.eye(3)).max() <= 4e-15
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.abs(a - b).max() <= 3 * rows * tol


def test_batch_matches_single():
    q = ss.SpinQuantumNumber.ONE
    sim = ss.Simulator(FIELD % "", q)
    sweep = np.array([[1e6, 0.0], [2e6, 0.0], [5e7, 0.0]])
    rows = np.array([100, 1, 333])
    out = sim.evaluate_batch(0.0, (rows + 0.5) * 1e-7, 1e-8, 1e-7, [1, 0, 0], sweep)
    for s in range(3):
        r = sim.evaluate(0.0, (rows[s] + 0.5) * 1e-7, 1e-8, 1e-7, [1, 0, 0], sweep[s])
        a, b = int(out.offsets[s]), int(out.offsets[s + 1])
        assert np.abs(np.asarray(out.time_evolution.cpu() if hasattr(out.time_evolution, "cpu")
                                 else out.time_evolution)[a:b] - r.time_evolution).max() <= 2e-14
