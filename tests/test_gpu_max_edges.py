"""The ordered maximum at the edges of its blocks (2048 values, strided over the threads): the first of equal zeros
is kept wherever the other one lies, a NaN anywhere never enters, and the initial value goes first."""

import numpy as np
import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


def fold(x, init):
    m = init
    for v in x:
        if v > m:
            m = v
    return m


@pytest.mark.parametrize("n", [1, 255, 256, 257, 2047, 2048, 2049, 4097, 600_000])
def test_gpu_max_edges(n):
    L = oppx.lib()
    rng = np.random.default_rng(n)
    out = torch.zeros(1, dtype=torch.float64, device="cuda")
    nb = int(L.oppx_max_scratch_bytes(n))
    scratch = torch.full((max(nb, 16),), 255, dtype=torch.uint8, device="cuda")
    for first, second in {(0, n - 1), (n - 1, 0), (n // 2, n // 3), (min(n - 1, 256), 0), (min(n - 1, 2048), n // 2)}:
        for values in ((0.0, -0.0), (-0.0, 0.0), (3.5, np.nan), (np.nan, np.nan)):
            x = -1.0 - rng.random(n)
            x[second], x[first] = values[1], values[0]
            for absv, init in ((0, -np.inf), (0, -0.0), (1, 0.0)):
                d = torch.from_numpy(x).cuda()
                oppx.check(L.oppx_max_reduce(n, d.data_ptr(), absv, init, out.data_ptr(), scratch.data_ptr(), nb,
                                             torch.cuda.current_stream().cuda_stream), "max_reduce")
                want = fold(np.abs(x) if absv else x, init) if n < 5000 else None
                got = float(out)
                if want is None:
                    live = (np.abs(x) if absv else x)
                    live = live[~np.isnan(live)]
                    top = live.max()
                    want = live[np.flatnonzero(live == top)[0]] if top > init else init
                assert got == want and np.signbit(got) == np.signbit(want), (first, second, values, absv, init)
