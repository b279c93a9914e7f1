"""The host build's spin-one steps without a quadratic shift (accumulated as
spin-half operators where the compiler sees the zero) against the same field with
a zero it cannot see."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss

FIELD = """__device__ void get_field(double t, const double* s, double* f)
{ f[0] = s[0] * cos(3e6 * t); f[1] = s[0] * sin(2e6 * t + 1); f[2] = s[0] * 0.7; %s }"""


@pytest.mark.parametrize("method", ["MAGNUS_CF4", "EULER", "HEUN"])
@pytest.mark.parametrize("frame", [True, False])
def test_rotation_matches_general(method, frame):
    sims = [ss.Simulator(FIELD % q, ss.SpinQuantumNumber.ONE, device=ss.Device.CPU, use_rotating_frame=frame,
                         integration_method=getattr(ss.IntegrationMethod, method)) for q in ("", "f[3] = s[1];")]
    dt, rows = 1e-8, 40
    for angle in (0.0, 1e-4, 0.012, 0.03, 0.3, 3.0):
        for fine in (1, 10, 1025, 2500):
            a, b = (s.evaluate(0.0, (rows + 0.5) * fine * dt, dt, fine * dt, [0.6, 0.0, 0.8j], [angle / dt, 0.0])
                    for s in sims)
            # up to 5000 factors, each rounded at the chunk residual's size (below 3)
            tol = 2e-15 + 2 * fine * 3 * 2.2e-16
            assert np.abs(a.time_evolution - b.time_evolution).max() <= tol
            assert np.abs(a.state - b.state).max() <= 3 * rows * tol
