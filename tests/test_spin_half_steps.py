"""Spin-half steps at the edges of their two series (0.018 and 1/4 rad), and
products longer than the block they are normalised after, against the closed
form of a constant field."""
from __future__ import annotations

import math

import numpy as np
import pytest

import spinsim_amd as ss

EPS = 2.0 ** -52
DEVICES = [ss.Device.CPU_SINGLE, pytest.param(ss.Device.ROCM, marks=pytest.mark.gpu)]
SRC = ("__device__ void get_field(double t, const double* s, double* f)\n"
       "{ f[0] = s[0]; f[1] = s[1]; f[2] = s[2]; }")


def closed_form(g):
    r = np.linalg.norm(g)
    n = g / r if r > 0 else g
    m = n[0] * np.array([[0, 1], [1, 0]]) + n[1] * np.array([[0, -1j], [1j, 0]]) + n[2] * np.diag([1, -1])
    return math.cos(r / 2) * np.eye(2) - 1j * math.sin(r / 2) * m


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("method", ["EULER", "MAGNUS_CF4"])
def test_constant_field(device, method):
    sim = ss.Simulator(SRC, ss.SpinQuantumNumber.HALF, device=device, use_rotating_frame=False,
                       integration_method=getattr(ss.IntegrationMethod, method),
                       lanes_per_step=None if device is ss.Device.CPU_SINGLE else 1)
    rng = np.random.default_rng(3)
    exponents = 1 if method == "EULER" else 2  # per step: CF4 halves the angle
    for r in (0.0, 1e-9, 0.0179, 0.0181, 0.249, 0.251, 3.0):
        for fine in (1, 2, 65536, 65537, 140000):
            if fine > 2 and r not in (0.0179, 0.251):
                continue
            g = rng.normal(size=3)
            g *= exponents * r / np.linalg.norm(g)
            u = sim.evaluate(0.0, 1.5 * fine, 1.0, float(fine), [1, 0], list(g)).time_evolution[0]
            # each step's angle is off by a few roundings, the same way every time
            bound = 16 * EPS * (1 + fine * exponents * r)
            assert np.abs(u - closed_form(fine * g)).max() <= bound, (r, fine)
            assert np.abs(u.conj().T @ u - np.eye(2)).max() <= 16 * EPS * (1 if r < 0.018 else fine)
