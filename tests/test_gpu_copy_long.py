"""oppx_copy_batch over more chunks than one launch may have workgroups: 32 GiB filled in 4-byte units (2 KiB a chunk), as
one job. Compared for equality."""

import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_blocks", [0, 1 << 25])
def test_gpu_copy_batch_of_more_chunks_than_workgroups(max_blocks):
    words = (1 << 33) + 4099  # 2^24 + 9 chunks: at 256 threads each a grid of more than 2^32 threads
    if torch.cuda.mem_get_info()[0] < 4 * words + (4 << 30):
        pytest.skip("less than 36 GiB of device memory free")
    x = torch.empty(words + 2, dtype=torch.int32, device="cuda")
    x[0] = x[-1] = -5
    assert x.data_ptr() % 8 == 0  # so that the row, one word on, moves in 4-byte units
    oppx.copy_batch([oppx.copy_job(x.data_ptr() + 4, 0, 4 * words, fill=7 | (11 << 32))],
                    torch.cuda.current_stream().cuda_stream, max_blocks)
    torch.cuda.synchronize()
    row = x[1:-1]
    step = 1 << 29
    for a in range(0, words, step):
        part = row[a:a + step]
        assert bool((part[0::2] == 7).all()) and bool((part[1::2] == 11).all()), a
    assert int(x[0]) == -5 and int(x[-1]) == -5
    del x, row, part
    torch.cuda.empty_cache()
