"""A callback's exp on the device, from the table's copy in LDS and from the
table itself: over table cells, at the ends of the range and beyond it."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss

pytestmark = pytest.mark.gpu

SOURCE = """
__device__ void get_field(double t, const double* sweep, double* field)
{ field[2] = (sweep[1] * exp(sweep[0])) * sweep[2]; }
"""


@pytest.mark.parametrize("head", ["", "#define SS_ADJ_AXES 7u\n"])
def test_exp_reads_its_table(head):
    rng = np.random.default_rng(5)
    node = np.arange(-1000, 1000) * (np.log(2) / 128)
    x = np.concatenate([node, node + np.log(2) / 256, rng.uniform(-708, 709, 500), [0.0, -0.0, -708.0, -720.0,
                        -740.0, -746.5, -1e6, -np.inf, 709.0, 709.7]])
    with np.errstate(under="ignore"):
        e = np.exp(x)
    # e * up * down is between 0.5 and 2, or 0: one radian at most
    down = np.where(e > 0, np.exp2(-np.floor(np.log2(np.where(e > 0, e, 1.0)) / 2)), 1.0)
    sweep = np.stack([x, down, down], axis=1)
    sim = ss.Simulator(head + SOURCE, ss.SpinQuantumNumber.HALF, use_rotating_frame=False,
                       integration_method=ss.IntegrationMethod.MIDPOINT_SAMPLE)
    plan = ss.BatchPlan(sim, 0.0, 1.5, 1.0, 1.0, np.array([1, 0]), sweep)
    plan.run()
    u = plan.u.cpu().numpy()[:, 0, 0]
    phase = (e * down) * down / 2
    # the exponential and its reference to an ulp each (a subnormal one to half
    # of its last place, 2^-1074), the step's sine and cosine to a few
    sub = np.where((e > 0) & (e < 2.3e-308), 5e-324 * down * down, 0.0)
    assert (np.abs(u - np.exp(-1j * phase)) <= 2e-15 + sub).all()
