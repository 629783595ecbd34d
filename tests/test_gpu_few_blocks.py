"""The move of a set of few blocks, whose first pass walks everything and adds its totals to the counters itself: up to the
last such size and past it, long walks (more evaluations than a larger set's first pass makes), both lane layouts and
block sizes, with removals; against the oracle's single walk. Charges: a node takes at most some 400 FP64 adds here, whose
order moves it by 400 * 2^-53 of their sum's size: 1e-12 of the largest node, as the other tests of the deposit allow."""

import numpy as np
import pytest

import oppx
import oracle

pytestmark = pytest.mark.gpu
DEFAULT = dict(tile=256, refill_min=16, split=0, persistent=0, sort_items=16, inline_hops=64,
               first_block=256, lanes=1)


@pytest.fixture(autouse=True)
def _restore_tuning():
    yield
    oppx.set_tuning(**DEFAULT)


@pytest.mark.parametrize("n,nx,cells,shape", [
    (1, 4, 2.0, {}), (257, 4, 1.0, {}), (5000, 30, 28.0, {}), (16_384, 12, 3.0, dict(lanes=4)), (16_385, 12, 3.0, dict(lanes=4)),
    (65_536, 16, 2.0, {}), (65_537, 16, 2.0, {}), (40_000, 14, 2.0, dict(first_block=1024)), (3000, 20, 15.0, dict(lanes=4)),
])
def test_gpu_move_of_few_blocks(n, nx, cells, shape):
    sigma = 0.02
    m = oppx.box_mesh(nx, nx, nx)
    ef = oppx.box_field_sines(m)
    pos, vel, p2c = oppx.box_particles(n, 17, sigma, m)
    dt = cells / nx / (sigma * np.sqrt(3.0))  # `cells` cells a step, no overlay
    oppx.set_tuning(**dict(DEFAULT, **shape))
    gpu, ref = oppx.FempicDevice(m, ef, pos, vel, p2c), oracle.FempicState(m, ef, pos, vel, p2c)
    gpu.work.fill_(255)
    gpu.counters[1:7] = 1234  # cleared by the step's begin, not by the move
    gpu.step_begin()
    faults = gpu.read_counters()["faults"]
    gpu.pass_fused(1e-3, 1.0, dt)
    got, hops = gpu.read_counters(), None
    other = oppx.FempicDevice(m, ef, pos, vel, p2c)
    other.push(1e-3, 1.0, dt)
    other.move()
    hops = other.hops[:n].cpu().numpy()
    gpu.holefill()
    ref.step(1e-3, 1.0, dt)
    out, exp = gpu.download(), ref.live()
    assert out["n"] == exp["n"] and got["removed"] == n - exp["n"] and got["faults"] == faults
    assert (got["max_hops"], got["total_hops"]) == (int(hops.max()), int(hops.sum()))
    if cells > 10:
        assert got["max_hops"] > 64
    for key in ("p2c", "pos", "vel", "lc"):
        assert np.array_equal(out[key], exp[key]), key
    assert np.abs(out["charge"] - exp["charge"]).max() <= 1e-12 * max(np.abs(exp["charge"]).max(), 1e-300)
