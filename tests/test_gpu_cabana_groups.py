"""The CabanaPIC deposit where the lanes of a wave split over cells in every way that changes the path: all in one
cell, two cells, shares at and just under the size from which a cell's lanes are summed in registers, more cells than
are summed so, single lanes, unordered cells, removed particles and a partial last wave.

An accumulator entry takes m <= 300 additions here; reordering them moves it by at most m * 2^-53 times the sum of the
terms' sizes, which is below 30 times the largest entry: 1e-12 of it. Positions, cells and hop counts are the oracle's
bits."""

import numpy as np
import pytest
import torch

import oracle
import oppx
from test_gpu_cabana import ACC_RTOL, CabanaDevice
from test_oracle_cabana import periodic_faces

pytestmark = pytest.mark.gpu
QSP, QDT_2MC, CDT = -0.01, 0.05, np.array([0.7, 0.6, 0.5])

# particles of consecutive cells; a wave is 64 consecutive particles
CASES = {
    "one": [64] * 30,
    "two": [32] * 40,
    "share": [56, 8, 57, 7, 8, 56, 7, 57, 63, 1, 1, 63] * 3,
    "three": [20, 22, 22] * 12,
    "eights": [8] * 90,
    "single": [1] * 200,
    "ragged": [300, 1, 7, 130, 9, 2, 65, 31] * 3 + [5],
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("form", ["ordered", "shuffled", "holes"])
def test_gpu_cabana_deposit_of_split_waves(name, form):
    rng = np.random.default_rng(len(name) * 31 + len(CASES[name]))
    dims = (6, 6, 6)
    nc = int(np.prod(dims))
    p2c = np.repeat(np.arange(len(CASES[name]), dtype=np.int32), CASES[name])
    n = p2c.size
    if form == "shuffled":
        rng.shuffle(p2c)
    interp = rng.normal(size=(nc, 18)) * np.array([0.5, 0.2, 0.2, 0.1] * 3 + [0.5, 0.2] * 3)
    pos, vel, weight = rng.uniform(-1, 1, (n, 3)), rng.normal(0, 0.4, (n, 3)), rng.uniform(0.5, 1.5, n)
    live = rng.random(n) < 0.8 if form == "holes" else np.ones(n, bool)
    c2c6 = periodic_faces(*dims)
    dev = CabanaDevice(dict(pos=pos, vel=vel, weight=weight, interp=interp, c2c6=c2c6, n_cells=nc,
                            p2c=np.where(live, p2c, np.int32(oppx.MAX_CELL_INDEX)).astype(np.int32)))
    opos, ovel, ow, oc = (np.ascontiguousarray(a[live]) for a in (pos, vel, weight, p2c))
    streak = np.zeros_like(opos)
    for _ in range(2):
        acc = np.zeros((nc, 12))
        hops = oracle.cabana_move_deposit(c2c6, interp, acc, opos, ovel, streak, ow, oc, QSP, QDT_2MC, CDT)
        tot, mx, faults = dev.step(QSP, QDT_2MC, CDT)
        assert faults == 0 and (tot, mx) == (int(hops.sum()), int(hops.max()))
        assert np.array_equal(dev.pos.cpu().numpy().T[live], opos) and np.array_equal(dev.vel.cpu().numpy().T[live], ovel)
        assert np.array_equal(dev.p2c.cpu().numpy()[live], oc) and np.array_equal(dev.hops.cpu().numpy()[live], hops)
        assert np.abs(dev.acc.cpu().numpy() - acc).max() <= ACC_RTOL * np.abs(acc).max()
