"""The FP64 deposit of blocks whose particles are in no order, through LDS copies of the charge: which blocks go that
way depends on their particles (ordered, in no order, half and half), on what the first pass hands over and on
the numbers of particles and nodes; every way gives the oracle's charge (1e-12 of the largest) and its particles."""

import numpy as np
import pytest

import oppx
import oracle

pytestmark = pytest.mark.gpu
DEFAULT = dict(tile=256, refill_min=16, split=0, persistent=0, sort_items=16, inline_hops=64, first_block=256, lanes=1)


@pytest.fixture(autouse=True)
def _restore_tuning():
    yield
    oppx.set_tuning(**DEFAULT)


@pytest.mark.parametrize("nx,n,shape", [
    (8, 262_143, {}), (8, 262_144, {}), (8, 300_001, dict(inline_hops=2)), (19, 270_000, {}), (20, 300_000, {}),
    (24, 500_063, {}), (25, 600_000, {}), (8, 270_000, dict(first_block=1024)), (8, 270_000, dict(lanes=4)),
])
@pytest.mark.parametrize("order", ["none", "cell", "half", "sparse"])
def test_gpu_dense_deposit(nx, n, shape, order):
    oppx.set_tuning(**dict(DEFAULT, **shape))
    sigma = 0.01
    m = oppx.box_mesh(nx, nx, nx)
    ef = oppx.box_field_sines(m)
    pos, vel, p2c = oppx.box_particles(n, nx, sigma, m)
    if order == "cell":
        pos, vel, p2c = oppx.sort_particles_by_cell(pos, vel, p2c)
    elif order == "half":
        h = n // 2
        pos[:h], vel[:h], p2c[:h] = oppx.sort_particles_by_cell(pos[:h], vel[:h], p2c[:h])
    elif order == "sparse":  # most of a block's particles are gone already
        p2c = np.where(np.arange(n) % 5 == 0, p2c, oppx.MAX_CELL_INDEX).astype(np.int32)
    dt = 0.5 / nx / (sigma * np.sqrt(3.0))
    bmin, bmax, gs = (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), 1.0 / (2 * nx)
    more = dict(overlay=oppx.dh_overlay(m, bmin, bmax, gs), bmin=bmin, bmax=bmax, gs=gs)
    start = np.where(p2c == oppx.MAX_CELL_INDEX, 0, p2c)
    gpu = oppx.FempicDevice(m, ef, pos, vel, start, **more)
    gpu.p2c[:n] = gpu.torch.from_numpy(p2c).cuda()
    here = p2c != oppx.MAX_CELL_INDEX
    ref = oracle.FempicState(m, ef, pos[here], vel[here], p2c[here], **more)
    for s in range(2):
        gpu.step_begin()
        gpu.pass_fused(1e-3, 1.0, dt, stage=s == 1)
        gpu.sort(drop_removed=True, lazy=s == 1) if s == 1 else gpu.holefill()
        r = ref.step(1e-3, 1.0, dt) if s == 0 else ref.step_sorted(1e-3, 1.0, dt)
        c = gpu.read_counters()
        if order != "sparse":  # (the hole fill leaves particles that were gone before the move where they are)
            assert c["size"] == r["size"]
        assert c["faults"] == 0 and c["total_hops"] == r["total_hops"] and c["max_hops"] == r["max_hops"]
        q = gpu.charge.cpu().numpy()
        assert np.abs(q - ref.charge).max() <= 1e-12 * np.abs(ref.charge).max()
        if order == "sparse":
            return
    out, exp = gpu.download(), ref.live()
    for key in ("p2c", "pos", "vel", "lc"):
        assert np.array_equal(out[key], exp[key]), key
