"""The table-driven sin and cos at the nodes and cell edges of the 1024-entry
table and on both sides of the reduction's limit, against numpy."""
from __future__ import annotations

import math

import numpy as np
import pytest

from spinsim_amd import host


@pytest.mark.parametrize("name,ref", [("sin", np.sin), ("cos", np.cos)])
def test_nodes_edges_and_limit(name, ref):
    j = np.arange(-3000, 3000)
    edge = (j + 0.5) * (math.tau / 1024)
    limit = 1e13 * (1 + np.arange(-40, 40) * 2.0 ** -50)
    x = np.concatenate([j * (math.tau / 1024), edge, np.nextafter(edge, 1e9), limit, -limit,
                        j * (math.tau / 1024) + 1e6])
    # both functions round to nearest up to about one ulp of 1
    assert np.abs(host.f64_eval(name, x) - ref(x)).max() <= 2.3e-16
