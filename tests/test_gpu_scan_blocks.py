"""The single-simulation scan on both sides of its workgroup counts: one, a
few and many totals before a workgroup, and the pass of its own beyond."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from spinsim_amd import _native

pytestmark = pytest.mark.gpu

ROWS_PER_BLOCK = 512


def _product(u):
    """u[n-1] ... u[0], by halves."""
    while len(u) > 1:
        if len(u) % 2:
            u = np.concatenate([u, np.eye(u.shape[1])[None]])
        u = u[1::2] @ u[0::2]
    return u[0]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("blocks,extra", [(1, 0), (2, -1), (256, 0), (256, 1), (257, 511), (512, 1), (513, 1),
                                          (768, 2), (1024, -1), (1024, 0), (1024, 1), (1300, 7)])
def test_states_follow_the_operators(dim, blocks, extra):
    n = blocks * ROWS_PER_BLOCK + extra
    rng = np.random.default_rng(blocks + dim)
    a = rng.normal(size=(64, dim, dim)) + 1j * rng.normal(size=(64, dim, dim))
    some = np.linalg.qr(a)[0]
    u = some[rng.integers(64, size=n)]
    psi = rng.normal(size=dim) + 1j * rng.normal(size=dim)
    psi /= np.linalg.norm(psi)
    lib = _native.lib()
    du = torch.as_tensor(u, device="cuda")
    state = torch.full((n, dim), float("nan"), dtype=torch.complex128, device="cuda")
    spin = torch.full((n, 3), float("nan"), dtype=torch.float64, device="cuda")
    size = lib.ss_state_scan_workspace(n, dim)
    work = torch.empty(size, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.ss_state_scan(psi.ctypes.data, du.data_ptr(), state.data_ptr(), spin.data_ptr(), n, dim,
                             work.data_ptr(), size, stream) == 0
    s = state.cpu().numpy()
    # about 40 products in a row, each within a few ulp of its unit columns
    assert np.array_equal(s[0], psi)
    assert np.abs(np.einsum("nij,nj->ni", u[:-1], s[:-1]) - s[1:]).max() <= 1e-13
    # the qr factors are unitary to an ulp or two: a product of n keeps its size to n ulp
    assert np.abs(_product(u[:-1]) @ psi - s[-1]).max() <= 1e-13 + 4 * n * 2.2e-16
    assert np.abs(spin.cpu().numpy()[-1, 2] - (abs(s[-1, 0]) ** 2 - abs(s[-1, -1]) ** 2)
                  * (0.5 if dim == 2 else 1.0)).max() <= 1e-14
