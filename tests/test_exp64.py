"""The field callbacks' table-driven float64 exp: at table nodes, cell edges,
the ends of its range and outside it, against the library function."""
from __future__ import annotations

import math

import numpy as np

from spinsim_amd import host


def test_within_an_ulp():
    rng = np.random.default_rng(7)
    node = np.arange(-130000, 130000, 37) * (math.log(2) / 128)
    edge = node + math.log(2) / 256
    x = np.concatenate([node, edge, np.nextafter(edge, 1e3), rng.uniform(-708, 709, 200000),
                        rng.uniform(-1, 1, 50000), [0.0, -0.0, 5e-324, -1e-300, -708.0, 709.0]])
    ref = np.exp(x)
    # 0.51 ulp of the table's form and the library's own rounding
    assert (np.abs(host.f64_eval("exp", x) - ref) <= np.spacing(ref)).all()
    assert np.mean(host.f64_eval("exp", x) == ref) > 0.95
    assert host.f64_eval("exp", [0.0])[0] == 1.0


def test_outside_the_range():
    x = np.array([-745.5, -745.2, -740.0, -709.0, -746.5, -1e9, -math.inf, 709.5, 709.9, 800.0,
                  math.inf, math.nan])
    with np.errstate(all="ignore"):
        np.testing.assert_array_equal(host.f64_eval("exp", x), np.exp(x))
