"""The hole fill where the most records move, a front half removed and a back half alive, at the sizes around which one
block or several fill; against the closed form: the k-th hole takes the k-th live record from the end."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 127, 128, 2048, 8191, 8192, 8193, 16_384, 300_001, 600_000])
@pytest.mark.parametrize("dims", [(3, 4, 1), (12, 1)])
def test_gpu_holefill_of_half_the_set(n, dims):
    L = oppx.lib()
    gone = torch.zeros(int(L.oppx_hole_bits_words(n)) * 64, dtype=torch.bool, device="cuda")
    gone[:n // 2] = True
    bits = (gone.reshape(-1, 64) * (torch.ones(1, dtype=torch.int64, device="cuda") << torch.arange(64, device="cuda"))).sum(1)
    dats = [(torch.arange(n, device="cuda")[None, :] + 3 * torch.arange(d, device="cuda")[:, None]).to(
        torch.float64 if q % 2 == 0 else torch.int32).contiguous() for q, d in enumerate(dims)]
    want = [t.flip(1) for t in dats]
    desc = (oppx.DatDesc * len(dats))(*[oppx.DatDesc(t.data_ptr(), t.shape[0], t.element_size()) for t in dats])
    ctr = torch.zeros(oppx.COUNTER_WORDS, dtype=torch.int32, device="cuda")
    ctr[0] = n
    scratch = torch.full((int(L.oppx_holefill_scratch_bytes(n)),), 255, dtype=torch.uint8, device="cuda")
    oppx.check(L.oppx_holefill(n, n, ctr.data_ptr(), bits.data_ptr(), desc, len(dats), scratch.data_ptr(),
                               scratch.numel(), torch.cuda.current_stream().cuda_stream), "holefill")
    size = n - n // 2  # an odd set's middle record stays
    assert ctr[:3].tolist() == [size, n // 2, n // 2]
    for t, w in zip(dats, want):
        assert torch.equal(t[:, :n // 2], w[:, :n // 2])
        if size > n // 2:
            assert torch.equal(t[:, n // 2], w[:, n // 2])
