"""The batch's step arithmetic on all simulations at once is evaluate()'s, value
for value, and keeps Python's errors for steps that have none."""
from __future__ import annotations

import numpy as np
import pytest

from spinsim_amd.batch import _batch_steps_one_by_one, batch_steps
from spinsim_amd.simulator import derive_steps


def test_same_values_as_one_by_one(capsys):
    rng = np.random.default_rng(6)
    n = 4000
    t0 = rng.uniform(-1e-3, 1e-3, n)
    dti = 10 ** rng.uniform(-9, -6, n)
    dto = np.where(rng.random(n) < 0.5, dti * rng.integers(1, 50, n), 10 ** rng.uniform(-9, -5, n))
    dto[:200] = dti[:200] * (rng.integers(0, 9, 200) + 0.5)  # halves round to even
    t1 = t0 + dto * rng.integers(0, 300, n) * rng.choice([1.0, 1 + 1e-15, 1 - 1e-15], n)
    t1 = np.maximum(t1, t0)
    _, dt, _, rows, fine = batch_steps(t0, t1, dti, dto, n)
    other = _batch_steps_one_by_one(t0, t1, dti, dto, n)
    assert np.array_equal(dt, other[0]) and np.array_equal(rows, other[1])
    assert np.array_equal(fine, other[2]) and fine.dtype == np.int32
    for s in range(0, n, 97):
        d, k, _ = derive_steps(t0[s], t1[s], dti[s], dto[s], warn=False)
        assert d == dt[s] and k == rows[s]
    assert f"{other[3]} simulation(s)" in capsys.readouterr().out


@pytest.mark.parametrize("dti,dto,error", [(0.0, 1e-6, ZeroDivisionError), (1e-7, 0.0, OverflowError),
                                           (float("nan"), 1e-6, ValueError),
                                           (1e-7, float("inf"), (ValueError, OverflowError))])
def test_errors(dti, dto, error):
    with pytest.raises(error):
        batch_steps(0.0, 1e-3, [1e-7, dti], [1e-6, dto], 2)


def test_end_before_start():
    with pytest.raises(ValueError):
        batch_steps([0.0, 1.0], 0.5, 1e-3, 1e-3, 2)
