"""Sines and cosines of a callback with many of them: the form that reduces large
arguments in line (float64 steps, 2/pi in 53-bit segments), from the first
argument beyond the table's reduction to the largest float64, and the registers
for whose sake it is taken."""
from __future__ import annotations

import math

import numpy as np
import pytest

import spinsim_amd as ss

pytestmark = pytest.mark.gpu

# s: 12 arguments (the compiler takes them to change with t), a weight each for
# cosine and sine, a zero
SOURCE = """
__device__ void get_field(double t, const double* s, double* f)
{
    double x = 0, y = 0;
    for (int k = 0; k < 12; ++k) {
        x += s[12 + k] * cos(s[k] + 0.0 * t) * exp(-s[36] * t * k);
        y += s[24 + k] * sin(s[k] + 0.0 * t) / (1 + s[36] * k * t);
    }
    f[2] = x + y;
}
"""
# float64 numbers next to multiples of pi / 2; the first is nearer to one, relative
# to pi / 2, than any other float64
NEAR = [math.ldexp(6381956970095103.0, 797), math.ldexp(6411027962775774.0, -48 + 60), 1e22]


def simulator(precision="fp64"):
    return ss.Simulator(SOURCE, ss.SpinQuantumNumber.HALF, use_rotating_frame=False, precision=precision)


def test_values():
    rng = np.random.default_rng(8)
    x = np.concatenate([1e13 * (1 + np.arange(-20, 20) * 2.0 ** -50), rng.uniform(1, 2, 2000) * 2.0 ** rng.integers(
        44, 1023, 2000), 2.0 ** np.arange(44, 1024), [2.0 ** 945 * (1 - 2.0 ** -53), 2.0 ** 54 + 4, 1.7976931348623157e308] + NEAR])
    x = np.concatenate([x, -x, rng.uniform(-1e6, 1e6, 200)])
    ref = np.array([[math.cos(v), math.sin(v)] for v in x])
    n = len(x)
    sweep = np.zeros((2 * n, 37))
    weight = np.maximum(1.0, 2.0 ** np.floor(-np.log2(np.abs(ref))))
    for part in (0, 1):
        rows, k = np.arange(part * n, part * n + n), np.arange(n) % 12
        sweep[rows, k] = x
        sweep[rows, 12 + 12 * part + k] = weight[:, part]
    plan = ss.BatchPlan(simulator(), 0.0, 1.5, 1.0, 1.0, np.array([1, 0]), sweep)
    plan.run()
    u = plan.u.cpu().numpy()[:, 0, 0].reshape(2, n).T
    # the table's functions round to 2.3e-16 of 1, relative to the value next to its
    # zeros; the reduction leaves 2^-104 quarter turns
    bound = 2e-15 + weight * 2.0 ** -103
    assert (np.abs(u - np.exp(-0.5j * weight * ref)) <= bound).all()


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_not_finite(value):
    sweep = np.zeros(37)
    sweep[3], sweep[15] = value, 1.0
    u = simulator().evaluate(0.0, 1.5, 1.0, 1.0, [1, 0], sweep).time_evolution
    assert np.isnan(u).any()


@pytest.mark.parametrize("precision", ["fp64", "fp32_bulk", "fp32"])
def test_registers(precision):
    """Three waves of the kernel fit a SIMD (512 registers a lane)."""
    sim = simulator(precision)
    sim.evaluate(0.0, 1.5, 1.0, 1.0, [1, 0], np.zeros(37))
    assert sim.module_info()["vgprs"] <= 168
