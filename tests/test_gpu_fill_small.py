"""The hole fill of a set that one block fills alone, up to its largest size and one past it, with a live count below the
host's bound, more components than one table holds, and an empty set; against the closed form: the k-th hole below the
new size takes the k-th live record from the end."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bound", [1, 64, 1025, 8191, 8192, 8193])
@pytest.mark.parametrize("live", ["all", "most", "none", "over"])
@pytest.mark.parametrize("frac,dims", [(0.0, (1,)), (0.02, (3, 3, 4, 1)), (0.5, (63, 1)), (0.97, (2, 64)), (1.0, (1,))])
def test_gpu_holefill_small(bound, live, frac, dims):
    L = oppx.lib()
    n = {"all": bound, "most": bound - bound // 5, "none": 0, "over": bound}[live]
    g = torch.Generator(device="cuda").manual_seed(bound + n)
    gone = torch.zeros(int(L.oppx_hole_bits_words(bound)) * 64, dtype=torch.bool, device="cuda")
    gone[:n] = torch.rand(n, device="cuda", generator=g) < frac
    bits = (gone.reshape(-1, 64) * (torch.ones(1, dtype=torch.int64, device="cuda") << torch.arange(64, device="cuda"))).sum(1)
    dats = [(torch.arange(bound, device="cuda")[None, :] + torch.arange(d, device="cuda")[:, None]).to(
        torch.float64 if q % 2 == 0 else torch.int32).contiguous() for q, d in enumerate(dims)]
    before = [t.clone() for t in dats]
    desc = (oppx.DatDesc * len(dats))(*[oppx.DatDesc(t.data_ptr(), t.shape[0], t.element_size()) for t in dats])
    ctr = torch.full((oppx.COUNTER_WORDS,), 5, dtype=torch.int32, device="cuda")
    ctr[0] = n if live != "over" else bound + 9  # a count past the bound is clamped to it
    scratch = torch.full((int(L.oppx_holefill_scratch_bytes(bound)),), 255, dtype=torch.uint8, device="cuda")
    oppx.check(L.oppx_holefill(bound, bound, ctr.data_ptr(), bits.data_ptr(), desc, len(dats), scratch.data_ptr(),
                               scratch.numel(), torch.cuda.current_stream().cuda_stream), "holefill")
    size = n - int(gone[:n].sum())
    holes = gone[:size].nonzero()[:, 0]
    source = ((~gone[size:n]).nonzero()[:, 0] + size).flip(0)
    c = ctr.tolist()
    assert (c[1], c[2]) == (n - size, holes.numel())
    assert c[0] == (size if size < n else n if live != "over" else bound + 9)
    for t, b in zip(dats, before):
        b[:, holes] = b[:, source]
        assert torch.equal(t[:, :size], b[:, :size])
