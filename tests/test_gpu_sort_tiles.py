"""The radix sort with every size of its tiles: which one a sort takes follows from the bound on the particles (4 keys a
thread below 2^20, 8 below 12 million, the tuned number from there on), so each is reached through such a bound, with
live counts at its edges, four digit passes, everything removed, one long run of equal keys and one full set; against a
stable argsort."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu
DEFAULT = dict(tile=256, refill_min=16, split=0, persistent=0, sort_items=16, inline_hops=64, first_block=256, lanes=1)


@pytest.fixture(autouse=True)
def _restore_tuning():
    yield
    oppx.set_tuning(**DEFAULT)


@pytest.mark.parametrize("items,bound", [(4, 1 << 20), (8, 1 << 20), (8, 12_000_000), (16, 12_000_000), (32, 12_000_000)])
@pytest.mark.parametrize("live,n_cells,removed", [(0, 7, 0.0), (1, 5, 0.0), (8191, 7, 0.0), (8193, 256, 0.1),
                                                  (4096, 100_000, 1.0), (20_000, 7, "run"), (70_001, 300, 0.3),
                                                  (300_000, 40_000_000, 0.1), ("all", 6_000_000, 0.02)])
def test_gpu_sort_tiles(items, bound, live, n_cells, removed):
    oppx.set_tuning(**dict(DEFAULT, sort_items=items))
    L = oppx.lib()
    live = bound if live == "all" else live
    stride = bound + 3
    g = torch.Generator(device="cuda").manual_seed(live + items)
    p2c = torch.randint(0, n_cells, (stride,), dtype=torch.int32, device="cuda", generator=g)
    if removed == "run":
        p2c[:] = 3
    else:
        p2c[torch.rand(stride, device="cuda", generator=g) < removed] = oppx.MAX_CELL_INDEX
    val = torch.randn((2, stride), dtype=torch.float64, device="cuda", generator=g)
    order = torch.argsort(p2c[:live], stable=True)
    gone = int((p2c[:live] == oppx.MAX_CELL_INDEX).sum())
    scratch = torch.full((int(L.oppx_sort_scratch_bytes(bound)),), 255, dtype=torch.uint8, device="cuda")
    desc = lambda ts: (oppx.DatDesc * len(ts))(*[oppx.DatDesc(t.data_ptr(), t.numel() // stride, t.element_size())
                                                 for t in ts])
    for lazy in (True, False):
        ctr = torch.full((oppx.COUNTER_WORDS,), 9, dtype=torch.int32, device="cuda")
        ctr[0] = live
        ins = [p2c] if lazy else [val, p2c]
        outs = [torch.full_like(t, -7) for t in ins]
        perm = torch.full((stride,), -7, dtype=torch.int32, device="cuda")
        oppx.check(L.oppx_sort_by_cell(bound, stride, ctr.data_ptr(), n_cells, p2c.data_ptr(), desc(ins), desc(outs),
                                       len(ins), perm.data_ptr(), 1, scratch.data_ptr(), scratch.numel(),
                                       torch.cuda.current_stream().cuda_stream), "sort")
        assert ctr[:3].tolist() == [live - gone, gone, 0]
        assert torch.equal(perm[:live].long(), order) and bool((perm[live:] == -7).all())
        for t, o in zip(ins, outs):
            assert torch.equal(o.reshape(-1, stride)[:, :live], t.reshape(-1, stride)[:, :live][:, order])
            assert bool((o.reshape(-1, stride)[:, live:] == -7).all())
