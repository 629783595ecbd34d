"""The two-pass move's block records and worklists: however much of a walk the first pass leaves to the walk pass
(blocks with empty, partly filled and full worklists, chunks of 8 and of 256 first-pass blocks, several rounds of
256 entries), the particles and the counters are those of the oracle's single walk."""

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


@pytest.mark.parametrize("n", [1, 255, 257, 5000, 70001])
@pytest.mark.parametrize("shape", [dict(inline_hops=1), dict(inline_hops=3), dict(inline_hops=16),
                                   dict(inline_hops=1, first_block=1024), dict(inline_hops=16, first_block=1024),
                                   dict(inline_hops=1, lanes=4), dict(inline_hops=17, lanes=4)])
def test_gpu_worklists_match_the_single_walk(n, shape):
    nx, sigma = 12, 0.02
    m = oppx.box_mesh(nx, nx, nx)
    ef = oppx.box_field_sines(m)
    pos, vel, p2c = oppx.box_particles(n, 31, sigma, m)
    dt = 3.0 / nx / (sigma * np.sqrt(3.0))  # three cells a step, no overlay: walks of up to some 30 evaluations
    oppx.set_tuning(**dict(DEFAULT, **shape))
    gpu = oppx.FempicDevice(m, ef, pos, vel, p2c)
    ref = oracle.FempicState(m, ef, pos, vel, p2c)
    gpu.work.fill_(255)  # the pass relies on nothing in its workspace
    gpu.step_begin()
    gpu.pass_fused(1e-3, 1.0, dt)
    got = gpu.read_counters()
    gpu.holefill()
    ref.step(1e-3, 1.0, dt)
    out, exp = gpu.download(), ref.live()
    assert out["n"] == exp["n"] and got["removed"] == n - exp["n"] and got["faults"] == 0
    for key in ("p2c", "pos", "vel", "lc"):
        assert np.array_equal(out[key], exp[key]), key
    assert np.abs(out["charge"] - exp["charge"]).max() <= 1e-12 * max(np.abs(exp["charge"]).max(), 1e-300)
    # the unfused loops' move clears the counters inside its first pass
    gpu2 = oppx.FempicDevice(m, ef, pos, vel, p2c)
    gpu2.counters[1:6] = 77
    gpu2.push(1e-3, 1.0, dt)
    gpu2.move()
    c = gpu2.read_counters()
    hops = gpu2.hops[:n].cpu().numpy()
    assert (c["removed"], c["holes_low"], c["faults"]) == (got["removed"], 0, 0)
    assert (c["max_hops"], c["total_hops"]) == (int(hops.max()), int(hops.sum()))
    assert (c["max_hops"], c["total_hops"]) == (got["max_hops"], got["total_hops"])
