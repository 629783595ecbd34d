"""Staged records back into the dats at the edges of the tile runs that an XCD takes (eighths, and runs of 64 tiles from
65,536 tiles on), with and without a permutation and with a live count below the bound; moved bits, compared for equality."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("live,bound", [(0, 1), (1, 1), (256, 256), (257, 5000), (8 * 256, 8 * 256), (8 * 256 + 1, 9 * 256),
                                        (100_003, 200_000), (65_536 * 256, 65_536 * 256), (65_536 * 256 + 1, 65_536 * 256 + 9),
                                        (65_536 * 256 + 512 * 256 + 77, 17_000_000)])
@pytest.mark.parametrize("permuted", [False, True])
def test_gpu_gather_records_edges(live, bound, permuted):
    rec = torch.arange(6 * bound, dtype=torch.float64, device="cuda")
    pos, vel = (torch.full((3, bound), -1.0, dtype=torch.float64, device="cuda") for _ in range(2))
    perm = torch.arange(bound, dtype=torch.int32, device="cuda").roll(1001) if permuted else None
    ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
    ctr[0] = live
    oppx.check(oppx.lib().oppx_gather_records(bound, bound, ctr.data_ptr(), perm.data_ptr() if permuted else None,
                                              rec.data_ptr(), pos.data_ptr(), vel.data_ptr(),
                                              torch.cuda.current_stream().cuda_stream), "gather_records")
    src = rec.reshape(bound, 6)[perm.long()] if permuted else rec.reshape(bound, 6)
    assert torch.equal(pos[:, :live], src[:live, :3].T) and torch.equal(vel[:, :live], src[:live, 3:].T)
    assert bool((pos[:, live:] == -1).all()) and bool((vel[:, live:] == -1).all()) and int(ctr[6]) == 0
