"""Hole fill at the edges of its word blocks, of its LDS table of block prefixes (sets past 67 M particles group
several blocks an entry) and of its component table (dats of more components than one launch moves), against the
closed form: the k-th hole below the new size takes the k-th live record from the end."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,frac,dims", [
    (1, 1.0, (1,)), (1, 0.0, (1,)), (63, 0.5, (3, 1)), (64, 0.02, (1, 4)), (65, 1.0, (2,)), (4097, 0.1, (3, 3, 4, 1)),
    (16383, 0.01, (3,)), (16384, 0.9, (1,)), (16385, 0.02, (63, 1)), (40000, 0.05, (65,)), (20000, 0.03, (40, 90, 2)),
    (67_108_865, 0.002, (1,)), (71_000_003, 0.3, (1,)),
])
def test_gpu_holefill_edges(n, frac, dims):
    L = oppx.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    gone = torch.rand(n, device="cuda", generator=g) < frac
    words = torch.zeros(int(L.oppx_hole_bits_words(n)) * 64, dtype=torch.bool, device="cuda")
    words[:n] = gone
    weight = torch.ones(1, dtype=torch.int64, device="cuda") << torch.arange(64, device="cuda")
    bits = (words.reshape(-1, 64) * weight).sum(1)
    dats, before = [], []
    for q, d in enumerate(dims):  # component d of record i holds i + d, in 8 and 4 bytes in turn
        t = torch.arange(n, device="cuda")[None, :] + torch.arange(d, device="cuda")[:, None]
        dats.append(t.to(torch.float64 if q % 2 == 0 else torch.int32).contiguous())
        before.append(dats[-1].clone())
    desc = (oppx.DatDesc * len(dats))(*[oppx.DatDesc(t.data_ptr(), t.shape[0], t.element_size()) for t in dats])
    ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
    ctr[0] = n
    scratch = torch.full((int(L.oppx_holefill_scratch_bytes(n)),), 255, dtype=torch.uint8, device="cuda")
    oppx.check(L.oppx_holefill(n, n, ctr.data_ptr(), bits.data_ptr(), desc, len(dats), scratch.data_ptr(),
                               scratch.numel(), torch.cuda.current_stream().cuda_stream), "holefill")
    size = n - int(gone.sum())
    holes = gone[:size].nonzero()[:, 0]
    source = ((~gone[size:]).nonzero()[:, 0] + size).flip(0)
    c = ctr.cpu()
    assert (int(c[0]), int(c[1]), int(c[2])) == (size, n - size, holes.numel())
    for t, b in zip(dats, before):
        b[:, holes] = b[:, source]
        assert torch.equal(t[:, :size], b[:, :size])
