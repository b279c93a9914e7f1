"""A quadratic shift that the callback sets in some steps only: whatever zeros the
compiler sees, no step is lost.  Against the same field plus a zero it cannot
see, for which every step takes the general form."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import spinsim_amd as ss

DEVICES = [ss.Device.CPU_SINGLE, pytest.param(ss.Device.ROCM, marks=pytest.mark.gpu)]
FRONT = ("__device__ void get_field(double t, const double* s, double* f)\n"
         "{ f[0] = 3e5 * cos(3e6 * t); f[1] = 2e5; f[2] = 4e5;\n  ")
# s: amplitude, switching times; the last is a zero the compiler cannot see
SHIFTS = {
    "if": "if (t > s[1]) f[3] = s[0];",
    "if_else": "if (t > s[1]) f[3] = s[0]; else f[3] = 0;",
    "ternary": "f[3] = t > s[1] ? s[0] : 0.0;",
    "return": "if (t < s[1]) return; f[3] = s[0];",
    "window": "if (t > s[1] && t < s[2]) f[3] = s[0];",
    "constant": "f[3] = 0; if (t > s[1]) f[3] = 1e5;",
    "switch": "switch ((int)(t / s[1])) { case 0: break; case 1: f[3] = s[0]; break; default: f[3] = 0; }",
    "loop": "for (int k = 1; k < 3; ++k) if (t > s[k]) f[3] = k * s[0];",
    "sweep": "if (s[0] > 0) f[3] = t > s[1] ? s[0] : 0.0;",
}
OPAQUE = {k: v.replace("return;", "{ f[3] = s[3]; return; }") + " f[3] += s[3];" for k, v in SHIFTS.items()}
METHODS = ["MAGNUS_CF4", "EULER", "HEUN"]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("form", sorted(SHIFTS))
@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("frame", [True, False])
def test_operators(device, form, method, frame):
    dt, fine, rows = 1e-8, 40, 12
    # switches inside output steps 3 and 7
    sweep = [2e5, 3.3 * fine * dt, 7.6 * fine * dt, 0.0]
    u = [ss.Simulator(FRONT + q[form] + " }", ss.SpinQuantumNumber.ONE, device=device, use_rotating_frame=frame,
                      integration_method=getattr(ss.IntegrationMethod, method))
         .evaluate(0.0, (rows + 0.5) * fine * dt, dt, fine * dt, [0.6, 0.0, 0.8j], sweep).time_evolution
         for q in (SHIFTS, OPAQUE)]
    # 80 factors, each rounded at the chunk residual's size (below 3)
    assert np.abs(u[0] - u[1]).max() <= 2e-15 + 80 * 3 * 2.2e-16


@pytest.mark.gpu
@pytest.mark.parametrize("form", sorted(SHIFTS))
@pytest.mark.parametrize("method", METHODS)
def test_gradients(form, method):
    dt, fine, rows = 1e-8, 40, 12
    sweep = [[2e5, 3.3 * fine * dt, 7.6 * fine * dt, 0.0]] * 2
    knots = np.linspace(0.0, rows * fine * dt, 7)
    amplitudes = np.random.default_rng(3).normal(0, 2e5, (2, 2, 7))
    grads = []
    for q in (SHIFTS, OPAQUE):
        sim = ss.ControlledSimulator(ss.SpinQuantumNumber.ONE, [ss.Control(a, knots) for a in "xy"],
                                     FRONT + q[form] + " }",
                                     integration_method=getattr(ss.IntegrationMethod, method))
        a = torch.tensor(amplitudes, device="cuda", requires_grad=True)
        psi = sim.final_state(a, 0.0, (rows + 0.5) * fine * dt, dt, fine * dt, [0.6, 0.0, 0.8], sweep)
        (1 - psi[:, -1].abs() ** 2).sum().backward()
        grads.append(a.grad.cpu().numpy())
    # both by the general derivative, rounded at each of 960 exponentials
    assert np.abs(grads[0] - grads[1]).max() <= 1e-12 * np.abs(grads[1]).max()
