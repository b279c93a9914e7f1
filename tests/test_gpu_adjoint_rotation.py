"""The backward pass without a quadratic shift (a rotation of three numbers)
against the general one (the series on state and costate) of the same pulses,
at the edges of its three ranges of angle."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import spinsim_amd as ss

pytestmark = pytest.mark.gpu

# the same field; the second sets q to a value the compiler cannot know is zero
PLAIN = "__device__ void get_field(double t, const double* s, double* f) { f[2] = s[0]; }"
GENERAL = ("__device__ void get_field(double t, const double* s, double* f) "
           "{ f[2] = s[0]; f[3] = s[1]; }")


# angle per exponential: inside 0.018, across it, across 1/2, beyond
@pytest.mark.parametrize("angle", [1e-3, 0.0179, 0.0181, 0.49, 0.51, 2.0])
@pytest.mark.parametrize("method", ["MAGNUS_CF4", "EULER", "HEUN"])
@pytest.mark.parametrize("frame", [True, False])
def test_rotation_matches_series(angle, method, frame):
    dt = 1e-7
    knots = np.linspace(0.0, 2e-6, 5)
    rng = np.random.default_rng(4)
    scale = angle / (dt * (0.5 if method != "EULER" else 1.0)) / math.sqrt(3)
    amplitudes = scale * rng.choice([-1.0, 1.0], (3, 3, 5)) * rng.uniform(0.98, 1.0, (3, 3, 5))
    grads = []
    for src in (PLAIN, GENERAL):
        sim = ss.ControlledSimulator(ss.SpinQuantumNumber.ONE,
                                     [ss.Control(a, knots) for a in "xyz"], src,
                                     use_rotating_frame=frame,
                                     integration_method=getattr(ss.IntegrationMethod, method))
        a = torch.tensor(amplitudes, device="cuda", requires_grad=True)
        psi = sim.final_state(a, 0.0, 2.05e-6, dt, 1e-6, [0.6, 0.0, 0.8], [[0.0, 0.0]] * 3)
        (1 - psi[:, -1].abs() ** 2).sum().backward()
        grads.append(a.grad.cpu().numpy())
    # the general derivative's series leaves out up to 2.4e-12 of each step's,
    # in sub-steps of at most 0.024; 40 exponentials of them
    assert np.abs(grads[0] - grads[1]).max() <= 1e-10 * np.abs(grads[1]).max()
