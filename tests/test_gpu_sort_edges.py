"""The radix sort at the edges of its tiles, row-scan chunks and XCD ranges: live counts below the bound (fewer
tiles than XCDs, none, one, a partial last tile), every tile size, one to four digit passes, with and without the
drop of removed particles, the permutation written directly or by the gather; against a stable argsort."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu
DEFAULT = dict(tile=256, refill_min=16, split=0, persistent=0, sort_items=16, inline_hops=64, first_block=256, lanes=1)


@pytest.fixture(autouse=True)
def _restore_tuning():
    yield
    oppx.set_tuning(**DEFAULT)


@pytest.mark.parametrize("items", [4, 8, 16, 32])
@pytest.mark.parametrize("live,bound,n_cells", [
    (0, 1, 5), (1, 1, 1), (1, 300_000, 300), (1023, 1024, 255), (1025, 4097, 256), (4096, 4096, 70_000),
    (32_769, 40_000, 65_535), (300_001, 2_000_000, 17_000_000), (5_000_000, 5_000_001, 1_000_003),
    (300_001, 1 << 20, 17_000_000), (9_000, 12_000_001, 255), (40_000, 12_000_000, 70_000),
    (1_300_000, 12_000_000, 1_000_003),  # the bounds from which a tile takes more keys per thread
])
def test_gpu_sort_edges(items, live, bound, n_cells):
    oppx.set_tuning(**dict(DEFAULT, sort_items=items))
    L = oppx.lib()
    g = torch.Generator(device="cuda").manual_seed(live + items)
    stride = bound + 3
    p2c = torch.randint(0, n_cells, (stride,), dtype=torch.int32, device="cuda", generator=g)
    p2c[torch.rand(stride, device="cuda", generator=g) < 0.1] = oppx.MAX_CELL_INDEX
    val = torch.randn((3, stride), dtype=torch.float64, device="cuda", generator=g)
    tag = torch.arange(stride, dtype=torch.int32, device="cuda")
    order = torch.argsort(p2c[:live], stable=True)
    gone = int((p2c[:live] == oppx.MAX_CELL_INDEX).sum())
    scratch = torch.full((int(L.oppx_sort_scratch_bytes(bound)),), 255, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    desc = lambda ts: (oppx.DatDesc * len(ts))(*[oppx.DatDesc(t.data_ptr(), t.numel() // stride, t.element_size())
                                                 for t in ts])
    for drop in (0, 1):
        for lazy in (True, False):
            ctr = torch.full((oppx.COUNTER_WORDS,), 9, dtype=torch.int32, device="cuda")
            ctr[0] = live
            ins = [p2c] if lazy else [val, tag, p2c]
            outs = [torch.full_like(t, -7) for t in ins]
            perm = torch.full((stride,), -7, dtype=torch.int32, device="cuda")
            oppx.check(L.oppx_sort_by_cell(bound, stride, ctr.data_ptr(), n_cells, p2c.data_ptr(), desc(ins), desc(outs),
                                           len(ins), perm.data_ptr(), drop, scratch.data_ptr(), scratch.numel(), stream),
                       "sort")
            c = ctr.cpu()
            assert (int(c[0]), int(c[1]), int(c[2])) == (live - gone if drop else live, gone, 0)
            assert torch.equal(perm[:live].long(), order) and bool((perm[live:] == -7).all())
            for t, o in zip(ins, outs):
                assert torch.equal(o.reshape(-1, stride)[:, :live], t.reshape(-1, stride)[:, :live][:, order])
                assert bool((o.reshape(-1, stride)[:, live:] == -7).all())
