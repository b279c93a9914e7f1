"""evaluate()'s routes -- sweep parameters in the kernel arguments or in a device
array, results in one copy, in several or left on the device -- give the same
bits; a capture refuses it."""
from __future__ import annotations

import numpy as np
import pytest

import spinsim_amd as ss
from spinsim_amd import _native
from spinsim_amd import simulator as S

pytestmark = pytest.mark.gpu

FIELD = """
__device__ void get_field(double t, const double* s, double* f)
{ f[0] = 2 * s[1] * cos(s[0] * t); f[1] = s[%d]; f[2] = s[0]; }
"""


@pytest.mark.parametrize("spin", ["HALF", "ONE"])
@pytest.mark.parametrize("rows", [0, 1, 300, 9000])
@pytest.mark.parametrize("lanes", [None, -2, 3])
def test_routes_agree(spin, rows, lanes):
    q = getattr(ss.SpinQuantumNumber, spin)
    sweep = [4.4e6, 1.3e4, 2e3] + [0.0] * (_native.SWEEP_INLINE - 3)
    results = []
    for size, where, limit in ((3, "numpy", None), (3, "torch", None), (3, "numpy", 0),
                               (_native.SWEEP_INLINE, "torch", None),
                               (_native.SWEEP_INLINE + 1, "torch", None),
                               (_native.SWEEP_INLINE + 1, "numpy", None)):
        sim = ss.Simulator(FIELD % 2, q)
        old = S.SINGLE_COPY_BYTES
        try:
            S.SINGLE_COPY_BYTES = old if limit is None else limit
            r = sim.evaluate(0.0, (rows + 0.5) * 1e-6, 1e-7, 1e-6, q.plus_x,
                             (sweep + [0.0])[:size], output=where, lanes_per_step=lanes)
        finally:
            S.SINGLE_COPY_BYTES = old
        arrays = [r.time, r.time_evolution, r.state, r.spin]
        results.append([a if isinstance(a, np.ndarray) else a.cpu().numpy() for a in arrays])
    assert results[0][1].shape == (rows, q.dimension, q.dimension)
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert np.array_equal(a, b)


def test_last_inline_parameter_is_read():
    n = _native.SWEEP_INLINE
    q = ss.SpinQuantumNumber.HALF
    sim = ss.Simulator(FIELD % (n - 1), q)
    runs = []
    for extra in ([], [0.0]):  # in the kernel arguments; in a device array
        sweep = [4.4e6, 1.3e4] + [0.0] * (n - 3) + [5e4] + extra
        runs.append(sim.evaluate(0.0, 1e-5, 1e-7, 1e-6, q.plus_z, sweep).time_evolution)
    assert np.array_equal(*runs) and abs(runs[0][0, 1, 0]) > 1e-3


def test_refused_while_capturing():
    import torch

    q = ss.SpinQuantumNumber.HALF
    sim = ss.Simulator(FIELD % 2, q)
    sim.evaluate(0.0, 1e-5, 1e-7, 1e-6, q.plus_z, [1.0, 2.0, 3.0], output="torch")
    x = torch.zeros(1, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1.0)
        with pytest.raises(RuntimeError, match="captured"):
            sim.evaluate(0.0, 1e-5, 1e-7, 1e-6, q.plus_z, [1.0, 2.0, 3.0], output="torch")
    for k in range(1, 3):
        graph.replay()
        torch.cuda.synchronize()
        assert x.item() == k
