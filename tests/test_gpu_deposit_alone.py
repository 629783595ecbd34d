"""The FP64 deposit by itself on either side of the size and the particles a cell from which a lane takes two particles,
with crowded tables, a live count below the bound, removed particles, cells out of range (counted as faults, not
deposited) and a partial last block; against sums in FP64 on the host. A node's charge is a sum of at most 4 n terms of
one sign, whose order moves it by far less than 1e-12 of the largest."""

import ctypes

import numpy as np
import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 18) + 1, 300_001])
@pytest.mark.parametrize("n_cells", [1, 3000, 131_072, 150_001])
@pytest.mark.parametrize("order", ["cells", "none"])
def test_gpu_deposit_alone(n, n_cells, order):
    rng = np.random.default_rng(n + n_cells)
    nn = max(4, n_cells // 5)
    c2n = rng.integers(0, nn, (n_cells, 4)).astype(np.int32)
    p2c = rng.integers(0, n_cells, n).astype(np.int32)
    if order == "cells":
        p2c.sort()
    gone = rng.random(n) < 0.03
    p2c[gone] = oppx.MAX_CELL_INDEX
    bad = rng.choice(np.flatnonzero(~gone), 5, replace=False)
    p2c[bad] = [n_cells, -1, n_cells + 7, -5, oppx.MAX_CELL_INDEX - 1]
    size = n - 77
    lc = rng.random((4, n))
    good = (p2c >= 0) & (p2c < n_cells) & (np.arange(n) < size)
    want = np.zeros(nn)
    np.add.at(want, c2n[p2c[good]].ravel(), lc[:, good].T.ravel())
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d = dict(lc=t(lc), p2c=t(p2c), c2n=t(c2n), charge=torch.zeros(nn, dtype=torch.float64, device="cuda"))
    ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
    ctr[0] = size
    parts = oppx.FempicParts(n, None, None, d["lc"].data_ptr(), d["p2c"].data_ptr())
    mesh = oppx.TetMesh(n_cells, nn, None, None, d["c2n"].data_ptr(), None)
    oppx.check(oppx.lib().oppx_fempic_deposit_atomic(n, ctypes.byref(parts), ctypes.byref(mesh), d["charge"].data_ptr(),
                                                     ctr.data_ptr(), torch.cuda.current_stream().cuda_stream), "deposit")
    assert int(ctr[6]) == int((bad < size).sum())
    assert np.abs(d["charge"].cpu().numpy() - want).max() <= 1e-12 * want.max()
