"""The gather of particle dats column by column: counts at the edges of its blocks, more columns than the grid holds side
by side, both element sizes, entries out of range (left untouched); moved bits are compared for equality."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("live,bound", [(0, 1), (1, 1), (255, 300), (1023, 5000), (1024, 1024), (1025, 1025), (8193, 9000),
                                        (70_001, 200_000)])
@pytest.mark.parametrize("dims", [(1,), (3, 1, 4), (63, 1), (70, 61)])
def test_gpu_gather_columns(live, bound, dims):
    stride = bound + 5
    g = torch.Generator(device="cuda").manual_seed(live + sum(dims))
    ins = [torch.randn((d, stride), dtype=torch.float64, device="cuda", generator=g) if k % 2 == 0 else
           torch.randint(0, 1 << 30, (d, stride), dtype=torch.int32, device="cuda", generator=g) for k, d in enumerate(dims)]
    outs = [torch.full_like(t, -7) for t in ins]
    perm = torch.randint(0, stride, (stride,), dtype=torch.int32, device="cuda", generator=g)
    perm[::97] = stride
    perm[5::113] = -1
    ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
    ctr[0] = live
    desc = lambda ts: (oppx.DatDesc * len(ts))(*[oppx.DatDesc(t.data_ptr(), t.shape[0], t.element_size()) for t in ts])
    oppx.check(oppx.lib().oppx_gather_dats(bound, stride, ctr.data_ptr(), perm.data_ptr(), desc(ins), desc(outs), len(ins),
                                           torch.cuda.current_stream().cuda_stream), "gather_dats")
    good = (perm >= 0) & (perm < stride) & (torch.arange(stride, device="cuda") < live)
    for t, o in zip(ins, outs):
        want = torch.where(good, t[:, perm.clamp(0, stride - 1).long()], torch.full_like(t, -7))
        assert torch.equal(o, want)
    assert int(ctr[0]) == live
