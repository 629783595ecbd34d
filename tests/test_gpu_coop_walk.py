"""The first pass's cooperative walk at its edges: waves with more and fewer moving lanes than the 32 records of a
fetch buffer, lanes that share a cell with their neighbour or with none, long and short walks in one wave, both block
sizes, removed particles in between; with and without an overlay, in place, through records and through a sort's
permutation. Particles, hop counts and counters equal the oracle's, bit for bit."""

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


@pytest.mark.parametrize("block", [256, 1024])
@pytest.mark.parametrize("n,order", [(1, "one"), (31, "one"), (64, "one"), (33, "own"), (64, "own"), (65, "pairs"),
                                     (1000, "one"), (1025, "pairs"), (5003, "own"), (20_011, "sorted")])
@pytest.mark.parametrize("overlay", [True, False])
def test_gpu_coop_walk(n, order, overlay, block):
    oppx.set_tuning(**dict(DEFAULT, first_block=block))
    nx, sigma = 9, 0.02
    m = oppx.box_mesh(nx, nx, nx)
    nc = m["n_cells"]
    rng = np.random.default_rng(n)
    if order == "one":  # every lane in one cell
        cell = np.full(n, nc // 2)
    elif order == "pairs":
        cell = np.repeat(rng.integers(0, nc, n // 2 + 1), 2)[:n]
    elif order == "own":  # unrelated cells
        cell = rng.integers(0, nc, n)
    else:
        cell = np.sort(rng.integers(0, nc, n))
    w = rng.dirichlet(np.ones(4), n)
    pos = (m["node_pos"][m["c2n"][cell]] * w[:, :, None]).sum(1)
    # some particles rest, some cross many cells
    vel = rng.normal(size=(n, 3)) * sigma * rng.choice([0.0, 1.0, 6.0], n)[:, None]
    p2c = cell.astype(np.int32)
    ef = oppx.box_field_sines(m)
    dt = 0.5 / nx / (sigma * np.sqrt(3.0))
    more = {}
    if overlay:
        bmin, bmax, gs = (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), 1.0 / 7
        more = dict(overlay=oppx.dh_overlay(m, bmin, bmax, gs), bmin=bmin, bmax=bmax, gs=gs)
    gpu = oppx.FempicDevice(m, ef, pos, vel, p2c, **more)
    ref = oracle.FempicState(m, ef, pos, vel, p2c, **more)
    for s in range(4):  # in place; records out; through the permutation, records out; through it, in place
        gpu.step_begin()
        gpu.pass_fused(1e-3, 1.0, dt, record_hops=True, stage=s in (1, 2))
        c = gpu.read_counters()
        if s in (1, 2):
            gpu.sort(drop_removed=True, lazy=True)
            r = ref.step_sorted(1e-3, 1.0, dt)
        else:
            gpu.holefill()
            r = ref.step(1e-3, 1.0, dt)
        assert c["faults"] == 0 and c["total_hops"] == r["total_hops"] and c["max_hops"] == r["max_hops"]
        assert gpu.read_counters()["size"] == r["size"]
        assert np.abs(gpu.charge.cpu().numpy() - ref.charge).max() <= 1e-12 * max(np.abs(ref.charge).max(), 1e-300)
    out, exp = gpu.download(), ref.live()
    assert out["n"] == exp["n"]
    for key in ("p2c", "pos", "vel", "lc"):
        assert np.array_equal(out[key], exp[key]), key
