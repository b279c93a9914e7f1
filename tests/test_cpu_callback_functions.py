"""HIP-C callbacks of the CPU devices that name library functions by namespace."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss

PULSE = ("__device__ void get_field(double t, const double* s, double* f)\n"
         "{ f[0] = 6e3 * %s(-t / 2e-5); f[1] = 0; f[2] = 1e4; }\n")


@pytest.mark.parametrize("call", ["exp", "::exp", "std::exp"])
def test_exponential_by_any_name(call):
    """The three calls name one function, so the results agree to its last bit."""
    head = "#include <cmath>\n" if call == "std::exp" else ""
    args = (0.0, 1e-4, 1e-6, 1e-5, np.array([1, 0], complex))
    runs = [ss.Simulator(src, ss.SpinQuantumNumber.HALF, ss.Device.CPU_SINGLE).evaluate(*args)
            for src in (PULSE % "exp", head + PULSE % call)]
    np.testing.assert_array_equal(runs[1].state, runs[0].state)
    # the pulse's area, 6e3 * 2e-5 (1 - e^-5) rad, about x with 1e4 rad/s about z
    assert 0 < abs(runs[0].state[-1, 1]) < 0.06
