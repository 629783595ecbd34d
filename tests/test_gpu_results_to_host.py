"""Both ways of a retired request's results to the host, the runtime's copy for long rows and one kernel for short ones: the
same bits whichever row takes which.

Bar: results bit-exact against the same request stepped alone."""

import pytest

import serve
from test_gpu_serve import alone, make_templates, same

pytestmark = pytest.mark.gpu

STEPS = 2


@pytest.mark.parametrize("long_row_bytes", [0, 4000, 30_000, 1 << 62])  # all, most, some and no rows by the runtime
def test_long_and_short_rows_arrive_alike(long_row_bytes):
    tpls = make_templates([(3, 4000), (4, 9000), (2, 700), (2, 1)], seed=67)
    arena = serve.FempicArena(max_cells=5000, max_nodes=2000, max_particles=40000, max_overlay=10000, max_insts=4)
    assert arena.long_row_bytes == 1 << 20
    arena.long_row_bytes = long_row_bytes
    slots = [arena.admit(t) for t in tpls]
    for _ in range(STEPS):
        arena.step()
    first = arena.retire_async(slots[1:3])
    arena.step()  # beside the copies
    for res, tpl in zip(first.wait(), tpls[1:3]):
        assert same(res, alone(tpl, STEPS))
    for res, tpl in zip(arena.retire([slots[0], slots[3]]), (tpls[0], tpls[3])):
        assert same(res, alone(tpl, STEPS + 1))
