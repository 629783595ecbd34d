"""The NESO step at the edges of its blocks (1024 threads, one or two particles a thread, a resident grid that strides)
and with quad records that are only 8-byte aligned, against the oracle, bit for bit; the directions a particle comes
with do not matter, removed particles are left alone."""

import numpy as np
import pytest
import torch

import oppx
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [True, False])
@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 2049, 524_289, 1_100_003])
def test_gpu_neso_edges(n, grid):
    nx, ny, cw, dt = 37, 23, 0.5, 0.5
    m = oppx.neso_mesh(nx, ny, cw)
    pos, vel, p2c = oppx.neso_particles(n, n, m, 4.0 * cw / dt)
    mdir = np.random.default_rng(n).integers(-1, 2, (n, 2)).astype(np.int32)
    gpu = oppx.NesoDevice(m, pos, vel, p2c, mdir=mdir, grid=grid)
    assert gpu.grid == grid
    if not grid:  # the records moved to an address that is 8 mod 16
        shifted = torch.zeros(gpu.cells.numel() + 1, dtype=torch.float64, device="cuda")
        shifted[1:] = gpu.cells
        gpu.cells = shifted[1:]
        assert gpu.cells.data_ptr() % 16 == 8
    gone = slice(n // 2, n // 2 + n // 10)
    gpu.p2c[gone] = oppx.MAX_CELL_INDEX
    gpu.step(dt, record_hops=True)
    c, out = gpu.read_counters(), gpu.download()
    op, om, oc = pos.copy(), mdir.copy(), p2c.copy()
    tot, hops = oracle.neso_step(n, nx, ny, cw, dt, m["c2c"], m["c_pos_ll"], op, vel, om, oc)
    om[gone], oc[gone], hops[gone] = mdir[gone], oppx.MAX_CELL_INDEX, 0
    assert np.array_equal(out["pos"], op) and np.array_equal(out["p2c"], oc)
    assert np.array_equal(out["mdir"], om) and np.array_equal(out["hops"], hops)
    assert (c["total_hops"], c["max_hops"], c["faults"]) == (int(hops.sum()), int(hops.max()), 0)
