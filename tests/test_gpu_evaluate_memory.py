"""Device memory of one evaluate(): results and the workspace of the launch that
follows, with a product per row only where that launch leaves them."""
from __future__ import annotations

import pytest
import torch

import spinsim_amd as ss
from spinsim_amd import _native

pytestmark = pytest.mark.gpu

SOURCE = """
__device__ void get_field(double t, const double* s, double* f)
{ f[0] = s[0] * cos(s[1] * t); f[2] = s[1]; }
"""


@pytest.mark.parametrize("spin", [ss.SpinQuantumNumber.HALF, ss.SpinQuantumNumber.ONE])
@pytest.mark.parametrize("precision,lanes,products", [
    ("fp64", None, True), ("fp64", 1, True), ("fp64", -2, False), ("fp64", 2, False),
    ("fp32_bulk", None, False), ("fp32", None, False), ("fp32", 1, True)])
def test_peak(spin, precision, lanes, products):
    n, d = 140000, spin.dimension  # (two lanes a step: 1094 workgroups)
    sim = ss.Simulator(SOURCE, spin, precision=precision)
    args = (0.0, (n + 0.5) * 2e-7, 1e-7, 2e-7, [1.0] + [0.0] * (d - 1), [1e4, 1e6])
    small = sim.evaluate(0.0, 4.5e-7, 1e-7, 2e-7, args[4], args[5], output="torch")
    del small
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    # (what is asked for: the allocator may give a block up to 1 MiB more)
    before = torch.cuda.memory_stats()["requested_bytes.all.current"]
    result = sim.evaluate(*args, output="torch", lanes_per_step=lanes)
    torch.cuda.synchronize()
    used = torch.cuda.memory_stats()["requested_bytes.all.peak"] - before
    results = n * (8 + 16 * d * d + 16 * d)
    scan = _native.lib().ss_state_scan_workspace(n, d)
    row = 16 * d * d
    if products:
        assert used <= results + n * row + (n // 4 + 1) * (row + 16 * d) + 4096
    else:
        assert used <= results + scan + 4096
    assert result.state.shape == (n, d)


@pytest.mark.parametrize("spin", [ss.SpinQuantumNumber.HALF, ss.SpinQuantumNumber.ONE])
def test_query(spin):
    """No launch needs less than it is given, or more than the largest."""
    sim = ss.Simulator(SOURCE, spin)
    lib, handle, d = _native.lib(), sim._module(torch.device("cuda", 0)).handle, spin.dimension
    for n in (1, 1000, 1024 * 256, 1024 * 256 + 1, 16384 * 256, 16384 * 256 + 1):
        scan, most = lib.ss_state_scan_workspace(n, d), lib.ss_evaluate_workspace(n, d)
        for lanes in (-64, -1, 0, 1, 2, 3, 33, 64):
            assert scan <= lib.ss_module_evaluate_workspace(handle, n, 1e-7, 1e-6, lanes) <= most
        assert lib.ss_module_evaluate_workspace(handle, n, 1e-7, 1e-6, -3) == scan
        assert (lib.ss_module_evaluate_workspace(handle, n, 1e-7, 1e-6, 1) == most)
    assert lib.ss_module_evaluate_workspace(handle, 0, 1e-7, 1e-6, 0) == 0
    assert lib.ss_module_evaluate_workspace(None, 10, 1e-7, 1e-6, 0) == 0
