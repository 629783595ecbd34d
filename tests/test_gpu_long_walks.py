"""Walks of tens of evaluations (starting cells unrelated to the positions, no overlay) in sets around the sizes at which
the first pass stops walking without a walk pass (65,536 particles), stops walking lane by lane to the end (196,608) and
hands long walks to many blocks of the walk pass instead; all or a few of the particles on such walks. Cells, weights,
positions, hops and counters bit-exact against the oracle, FP64 deposit within 1e-12 relative."""

import numpy as np
import pytest

import oppx
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65_536, 65_537, 196_608, 196_609, 270_001])
@pytest.mark.parametrize("share", [1.0, 0.02])
@pytest.mark.parametrize("fused", [True, False])
def test_gpu_long_walks(n, share, fused):
    nx = 26  # 105,456 tets, 19,683 nodes: no LDS copies of the charge; walks of up to some 170 evaluations
    m = oppx.box_mesh(nx, nx, nx)
    ef = oppx.box_field_sines(m)
    pos, vel, p2c = oppx.box_particles(n, 7, 0.01, m)
    rng = np.random.default_rng(n)
    far = rng.random(n) < share
    p2c[far] = rng.integers(0, m["n_cells"], int(far.sum()))
    gpu = oppx.FempicDevice(m, ef, pos, vel, p2c)
    ref = oracle.FempicState(m, ef, pos, vel, p2c)
    dt = 0.2 / nx / (0.01 * np.sqrt(3.0))
    if fused:
        gpu.step_begin()
        gpu.pass_fused(1e-3, 1.0, dt, record_hops=True)
        gpu.holefill()
    else:
        gpu.step_unfused(1e-3, 1.0, dt)
    r = ref.step(1e-3, 1.0, dt)
    c = gpu.read_counters()
    assert c["faults"] == 0 and r["max_hops"] > 64
    assert (c["size"], c["total_hops"], c["max_hops"]) == (r["size"], r["total_hops"], r["max_hops"])
    out, exp = gpu.download(), ref.live()
    for key in ("p2c", "pos", "vel", "lc"):
        assert np.array_equal(out[key], exp[key]), key
    assert np.abs(out["charge"] - exp["charge"]).max() <= 1e-12 * np.abs(exp["charge"]).max()
