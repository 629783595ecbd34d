"""The FP32 deposit's run sums at the edges of its tiles of 2048 particles and windows of 64 more, and of the length
(64) from which a wave sums a run: bit for bit a NumPy restatement of the documented order (one lane a run, or 64
lane sums added in lane order), read in place, through a permutation, and with the sorted FP32 copy."""

import numpy as np
import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu
f32 = np.float32


def kahan(rows):
    s, c = np.zeros(rows.shape[1], f32), np.zeros(rows.shape[1], f32)
    for x in rows:
        y = x - c
        t = s + y
        c = (t - s) - y
        s = t
    return s


def run_sum(rows):
    if len(rows) <= 64:
        return kahan(rows)
    # lane l: particles l, l + 64, ...: the rounds of all lanes are one array, short lanes padded by nothing
    lanes = np.stack([kahan(rows[l::64]) for l in range(64)])
    return kahan(lanes)


CASES = {
    "empty": [], "one": [1], "tile": [2048], "tile_and_one": [2049], "window": [2112], "past_window": [2113],
    "around_64": [63, 64, 65, 66, 1, 64, 65], "end_on_tile": [64] * 32 + [5], "cross_64": [2000] + [64, 65, 3],
    "cross_short": [2047, 1, 1, 2], "cross_long": [1985, 127, 63, 64], "starts_at_edge": [2048, 64, 1983, 65, 65],
    "ones": [1] * 4200, "three_tiles": [6000, 2, 200],
}


@pytest.mark.parametrize("removed", [0, 7])
@pytest.mark.parametrize("name", list(CASES))
def test_gpu_run_sums_at_edges(name, removed):
    rng = np.random.default_rng(len(name))
    runs = CASES[name]
    # runs of increasing cells with gaps; every cell has four nodes of its own and one they all share
    cells = np.cumsum(rng.integers(1, 4, len(runs))) if runs else np.zeros(0, int)
    n_cells = int(cells[-1]) + 3 if runs else 5
    p2c = np.concatenate([np.repeat(cells, runs), np.full(removed, oppx.MAX_CELL_INDEX)]).astype(np.int32)
    n, cap = len(p2c), len(p2c) + 5
    lc = rng.random((4, cap))
    start = np.arange(0, 4 * n_cells + 1, dtype=np.int32)
    ref = np.arange(4 * n_cells, dtype=np.int32)
    want = np.zeros((n_cells, 4), f32)
    at = 0
    for c, k in zip(cells, runs):
        want[c] = run_sum(lc[:, at:at + k].T.astype(f32))
        at += k
    want = kahan(want.reshape(1, -1))  # a node of one partial: 0 + partial

    L = oppx.lib()
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    perm = np.concatenate([rng.permutation(n), np.arange(n, cap)]).astype(np.int32)
    moved = lc.copy()
    moved[:, perm[:n]] = lc[:, :n]  # lc in the order before the sort
    pad = np.full(cap, 3, np.int32)
    pad[:n] = p2c
    d = dict(p2c=t(pad), lc=t(lc), moved=t(moved), perm=t(perm), start=t(start), ref=t(ref))
    part = torch.full((4 * n_cells,), 9.0, device="cuda")
    scratch = torch.full((int(L.oppx_fempic_deposit_scratch_bytes(cap)),), 255, dtype=torch.uint8, device="cuda")
    copy = torch.zeros(4 * cap, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for form in ("place", "perm", "copy"):
        ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
        ctr[0] = n
        out = torch.full((4 * n_cells,), 5.0, device="cuda")
        tail = (n_cells, d["start"].data_ptr(), None, d["ref"].data_ptr(), 4 * n_cells, part.data_ptr(), None,
                out.data_ptr(), scratch.data_ptr(), scratch.numel(), stream)
        if form == "place":
            rc = L.oppx_fempic_deposit_sorted_f32(cap, cap, ctr.data_ptr(), d["p2c"].data_ptr(), d["lc"].data_ptr(), *tail)
        else:
            rc = L.oppx_fempic_deposit_sorted_f32_perm(cap, cap, ctr.data_ptr(), d["p2c"].data_ptr(),
                                                       d["moved"].data_ptr(), d["perm"].data_ptr(),
                                                       copy.data_ptr() if form == "copy" else None, *tail)
        oppx.check(rc, form)
        assert int(ctr[6]) == 0, form
        assert np.array_equal(out.cpu().numpy(), want.ravel()), form
    if len(runs) > 2:  # not sorted: counted, never silent
        bad = pad.copy()
        bad[:n - removed] = bad[:n - removed][::-1]
        ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
        ctr[0] = n
        oppx.check(L.oppx_fempic_deposit_sorted_f32(cap, cap, ctr.data_ptr(), t(bad).data_ptr(), d["lc"].data_ptr(),
                                                    *tail), "unsorted")
        assert int(ctr[6]) == len(runs) - 1
