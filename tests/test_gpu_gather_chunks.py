"""The gather of particle dats whose results are past the 256 MB cache: an XCD takes its tiles in chunks of 512 (4,194,304
live particles to a full one), on at most 2^18 workgroups that stride over chunks and columns; counts at a chunk's edge, more
columns than the grid holds side by side, a live count far below the bound, entries out of range (left untouched). Moved
bits are compared for equality."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu
CHUNK = 512 * 8 * 1024


@pytest.mark.parametrize("live,bound,dims", [
    (CHUNK - 1, CHUNK + 9, (3, 1, 6)), (CHUNK, CHUNK, (3, 1, 6)), (CHUNK + 1, CHUNK + 1, (3, 1, 6)),  # one chunk, then two
    (2 * CHUNK + 8 * 1024 + 1, 9_000_000, (4,)),      # a third chunk of two tiles an XCD
    (5_000_000, 5_000_000, (0, 40)), (1_000, 5_000_000, (0, 40)), (0, 5_000_000, (0, 40)),  # 40 columns: the grid strides
    (5_000_000, 5_000_001, (1, 70)),                  # 71 columns, 64 of them side by side
])
def test_gpu_gather_in_chunks(live, bound, dims):
    stride = bound + 5
    g = torch.Generator(device="cuda").manual_seed(live + sum(dims))
    ins = [torch.randn((d, stride), dtype=torch.float64, device="cuda", generator=g) if k % 2 == 0 else
           torch.randint(0, 1 << 30, (d, stride), dtype=torch.int32, device="cuda", generator=g)
           for k, d in enumerate(dims) if d]
    assert bound * sum(t.shape[0] * t.element_size() for t in ins) > 256 << 20
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
    at = perm.clamp(0, stride - 1).long()
    for t, o in zip(ins, outs):
        for col in range(t.shape[0]):
            assert torch.equal(o[col], torch.where(good, t[col][at], torch.full_like(t[col], -7))), col
    assert int(ctr[0]) == live
