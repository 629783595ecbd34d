"""oppx_copy_batch against numpy: rows of every alignment and remainder, fills, rebased index records, more rows than one
launch takes, rows of several blocks, pinned memory. Bytes are moved, so everything is compared for equality."""

import numpy as np
import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu
MAX = oppx.MAX_CELL_INDEX


def run(jobs, max_blocks=0):
    oppx.copy_batch(jobs, torch.cuda.current_stream().cuda_stream, max_blocks)
    torch.cuda.synchronize()


@pytest.mark.parametrize("words", [1, 2, 3, 4, 5, 7, 2047, 2048, 2049, 4096, 70_001])
@pytest.mark.parametrize("to,frm", [(0, 0), (2, 2), (4, 2), (1, 1), (3, 0), (0, 1)])
@pytest.mark.parametrize("rows,blocks", [(1, 0), (3, 5), (40, 0), (40, 1)])
def test_gpu_copy_batch_rows(words, to, frm, rows, blocks):
    if rows * words > 300_000:
        rows = 4
    rng = np.random.default_rng(words + 7 * to + frm)
    ds, ss = words + to + 5, words + frm + 2
    src = rng.integers(-2**31, 2**31, rows * ss + 8, dtype=np.int64).astype(np.int32)
    a, b = torch.from_numpy(src).cuda(), torch.full((rows * ds + 8,), 77, dtype=torch.int32, device="cuda")
    run([oppx.copy_job(b.data_ptr() + 4 * to, a.data_ptr() + 4 * frm, 4 * words, rows, 4 * ds, 4 * ss)], blocks)
    want = np.full(rows * ds + 8, 77, np.int32)
    for r in range(rows):
        want[to + r * ds:to + r * ds + words] = src[frm + r * ss:frm + r * ss + words]
    assert np.array_equal(b.cpu().numpy(), want)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 513, 2050])
@pytest.mark.parametrize("rec", [(1, 0, 1), (2, 1, 1), (8, 2, 4), (128, 3, 120)])
@pytest.mark.parametrize("shift,in_place,pinned", [(0, False, False), (1, False, True), (2, True, False), (0, True, False)])
def test_gpu_copy_batch_rebases_like_offset_indices(n, rec, shift, in_place, pinned):
    words = n * rec[0]
    rng = np.random.default_rng(words + shift)
    src = rng.integers(-3, 1000, words + 4, dtype=np.int64).astype(np.int32)
    src[rng.random(words + 4) < 0.1] = MAX
    a = torch.from_numpy(src).cuda()
    b = a if in_place else torch.zeros(words + 4, dtype=torch.int32, device="cpu" if pinned else "cuda", pin_memory=pinned)
    run([oppx.copy_job(b.data_ptr() + 4 * shift, a.data_ptr() + 4 * shift, 4 * words, add=12_345, rec=rec)])
    want = src[shift:shift + words].copy().reshape(n, rec[0])
    part = want[:, rec[1]:rec[1] + rec[2]]
    part[(part >= 0) & (part != MAX)] += 12_345
    assert np.array_equal(b.cpu().numpy()[shift:shift + words], want.ravel())


def test_gpu_copy_batch_mixes_fills_and_copies_in_one_call():
    n = 50
    src = torch.arange(3 * n, dtype=torch.float64, device="cuda")
    out = torch.full((n, 33), -1.0, dtype=torch.float64, device="cuda")
    jobs, want = [], out.cpu().numpy()
    for i in range(n):
        w = i % 30
        if i % 3 == 0:
            jobs.append(oppx.copy_job(out[i].data_ptr(), 0, 8 * w, fill=int(np.float64(i).view(np.uint64))))
            want[i, :w] = i
        else:
            jobs.append(oppx.copy_job(out[i].data_ptr(), src.data_ptr() + 8 * i, 8 * w))
            want[i, :w] = np.arange(i, i + w)
    run(jobs)
    assert np.array_equal(out.cpu().numpy(), want)
    word = torch.zeros(7, dtype=torch.int32, device="cuda")
    run([oppx.copy_job(word.data_ptr() + 4, 0, 20, fill=(5 << 32) | 9)])
    assert word.tolist() == [0, 9, 5, 9, 5, 9, 0]
    run([])


@pytest.mark.parametrize("bad", [dict(nbytes=-4), dict(nbytes=6), dict(dst=0), dict(dst=2), dict(rows=2, dst_stride=4),
                                 dict(rows=2, dst_stride=8, src_stride=4), dict(add=1, rec=(3, 0, 1)),
                                 dict(add=1, rec=(8, 6, 3)), dict(add=1, rec=(256, 0, 1)), dict(rows=-1)])
def test_gpu_copy_batch_refuses(bad):
    a = torch.zeros(64, dtype=torch.int32, device="cuda")
    job = dict(dst=a.data_ptr(), src=a.data_ptr() + 128, nbytes=8)
    job.update({k: v for k, v in bad.items() if k != "dst"})
    if "dst" in bad:
        job["dst"] = bad["dst"] and a.data_ptr() + bad["dst"]
    with pytest.raises(RuntimeError):
        run([oppx.copy_job(**job)])


def test_gpu_results_dropped_before_their_copies_end():
    """A pinned block goes back to the host allocator only when nothing writes it any more."""
    import serve
    from workloads import box_instance
    arena = serve.FempicArena(20_000, 10_000, 60_000, 40_000, 8)
    tpl = serve.Template.of(box_instance(6, 20_000, 3, 0.01)).make_resident()
    for _ in range(3):
        slot = arena.admit(tpl)
        arena.step()
        pend = arena.retire_async([slot])
        done = pend.events
        del pend
        assert all(e.query() for e in done)
