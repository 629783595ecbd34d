"""The FP64 deposit's LDS table with node sets that crowd it: nodes that share a line, lines that share a group, more
distinct nodes in a block than the table has slots, few nodes added to by every particle; against sums in FP64 on
the host (1e-12 of the largest charge: the order of the additions differs)."""

import ctypes

import numpy as np
import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 1023, 4099, 60_000])
@pytest.mark.parametrize("nodes", ["one", "line", "strided", "spread", "all_distinct"])
def test_gpu_deposit_table(n, nodes):
    rng = np.random.default_rng(n)
    nn = 1 << 20
    if nodes == "one":
        c2n = np.full((n, 4), 12345)
    elif nodes == "line":  # 64 nodes: four lines
        c2n = 4096 + rng.integers(0, 64, (n, 4))
    elif nodes == "strided":  # one node a line, lines 64 apart
        c2n = 1024 * rng.integers(0, 1000, (n, 4)) + 7
    elif nodes == "spread":
        c2n = rng.integers(0, nn, (n, 4))
    else:  # every add of a block to a node of its own
        c2n = (np.arange(4 * n).reshape(n, 4) * 17) % nn
    c2n = c2n.astype(np.int32)
    lc = rng.random((4, n))
    p2c = np.arange(n, dtype=np.int32)
    p2c[rng.random(n) < 0.1] = oppx.MAX_CELL_INDEX
    live = p2c != oppx.MAX_CELL_INDEX
    want = np.zeros(nn)
    np.add.at(want, c2n[live].ravel(), lc[:, live].T.ravel())
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d = dict(lc=t(lc), p2c=t(p2c), c2n=t(c2n), charge=torch.zeros(nn, dtype=torch.float64, device="cuda"))
    ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
    ctr[0] = n
    parts = oppx.FempicParts(n, None, None, d["lc"].data_ptr(), d["p2c"].data_ptr())
    mesh = oppx.TetMesh(n, nn, None, None, d["c2n"].data_ptr(), None)
    oppx.check(oppx.lib().oppx_fempic_deposit_atomic(n, ctypes.byref(parts), ctypes.byref(mesh), d["charge"].data_ptr(),
                                                     ctr.data_ptr(), torch.cuda.current_stream().cuda_stream), "deposit")
    got = d["charge"].cpu().numpy()
    assert int(ctr[6]) == 0
    assert np.abs(got - want).max() <= 1e-12 * max(want.max(), 1e-300)
    assert not got[want == 0].any()
