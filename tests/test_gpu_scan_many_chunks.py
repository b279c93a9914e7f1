"""Batch scans around the number of chunks from which a thread takes one row in
the second pass, against the same scans in chunks of 4096 rows."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from spinsim_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,layout", [(2, 0), (2, 1), (2, 2), (3, 0)])
@pytest.mark.parametrize("total", [524288, 524289, 700001, 2097151])
def test_passes_agree(dim, layout, total):
    lib = _native.lib()
    rng = np.random.default_rng(total)
    cuts = np.sort(rng.integers(0, total + 1, size=300))
    offsets = np.concatenate([[0, 0], cuts, [total]]).astype(np.int64)  # empty ones among them
    sims = len(offsets) - 1
    a = rng.normal(size=(total, 2)) + 1j * rng.normal(size=(total, 2))
    a /= np.linalg.norm(a, axis=1)[:, None]
    if dim == 2:
        u = np.stack([a[:, 0], -a[:, 1].conj(), a[:, 1], a[:, 0].conj()], axis=1).reshape(total, 2, 2)
        stored = np.ascontiguousarray(a) if layout == 1 else u
    else:
        some = np.linalg.qr(rng.normal(size=(64, 3, 3)) + 1j * rng.normal(size=(64, 3, 3)))[0]
        stored = some[rng.integers(64, size=total)]
    psi = rng.normal(size=(sims, dim)) + 1j * rng.normal(size=(sims, dim))
    psi /= np.linalg.norm(psi, axis=1)[:, None]
    du, dpsi, off = (torch.as_tensor(x, device="cuda") for x in (stored, psi, offsets))
    stream = torch.cuda.current_stream().cuda_stream
    got = {}
    for chunk in (1024, 4096):
        size = lib.ss_batch_scan_workspace(total, dim, chunk)
        work = torch.empty(size, dtype=torch.uint8, device="cuda")
        state = torch.full((total, dim), float("nan"), dtype=torch.complex128, device="cuda")
        back = state.clone()
        spin = torch.full((total, 3), float("nan"), dtype=torch.float64, device="cuda")
        assert lib.ss_batch_state_scan(dpsi.data_ptr(), du.data_ptr(), state.data_ptr(), spin.data_ptr(),
                                       off.data_ptr(), sims, total, dim, chunk, layout, work.data_ptr(), size,
                                       stream) == 0
        if layout == 0:
            assert lib.ss_batch_costate_scan(dpsi.data_ptr(), du.data_ptr(), back.data_ptr(), off.data_ptr(), sims,
                                             total, dim, chunk, work.data_ptr(), size, stream) == 0
        got[chunk] = [x.cpu().numpy() for x in (state, spin, back)]
    # the same products of at most `total` unitary factors in another order:
    # their norms wander by the factors' own rounding, in both alike
    tol = 1e-13 + 2e-15 * np.sqrt(total)
    for x, y in zip(got[1024][:2 if layout else 3], got[4096]):
        assert np.isfinite(x).all() and np.abs(x - y).max() <= tol
