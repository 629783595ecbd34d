"""The NESO step at the sizes where its blocks and its grid change (16,384, 65,536 and 6 million particles), with the records
of the periodic grid computed and gathered, against the oracle, bit for bit."""

import numpy as np
import pytest

import oppx
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [True, False])
@pytest.mark.parametrize("n", [16_383, 16_384, 65_535, 65_536, 5_999_999, 6_000_000])
def test_gpu_neso_blocks(n, grid):
    nx, ny, cw, dt = 61, 40, 0.5, 0.5
    m = oppx.neso_mesh(nx, ny, cw)
    pos, vel, p2c = oppx.neso_particles(n, n, m, 2.0 * cw / dt)
    gpu = oppx.NesoDevice(m, pos, vel, p2c, grid=grid)
    assert gpu.grid == grid
    gpu.step(dt, record_hops=True)
    c, out = gpu.read_counters(), gpu.download()
    om = np.ones((n, 2), np.int32)
    tot, hops = oracle.neso_step(n, nx, ny, cw, dt, m["c2c"], m["c_pos_ll"], pos, vel, om, p2c)
    assert np.array_equal(out["pos"], pos) and np.array_equal(out["p2c"], p2c)
    assert np.array_equal(out["mdir"], om) and np.array_equal(out["hops"], hops)
    assert (c["total_hops"], c["max_hops"], c["faults"]) == (int(hops.sum()), int(hops.max()), 0)
