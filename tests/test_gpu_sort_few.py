"""The sort of few tiles, whose scatters sum the tiles' digit counts themselves: tile counts at the batch of counts in
flight and at the last such size, live counts below the bound, one to four digit passes; against a stable argsort."""

import pytest

import test_gpu_sort_edges as edges
from test_gpu_sort_edges import _restore_tuning  # noqa: F401  (the fixture puts the tuning back)

pytestmark = edges.pytestmark


@pytest.mark.parametrize("n_cells", [200, 255, 256, 65_535, 1 << 20, 20_000_000])
@pytest.mark.parametrize("live,bound", [(0, 1024), (1024, 1024), (31 * 1024 + 1, 32 * 1024), (32 * 1024 + 1, 40_000),
                                        (33 * 1024, 33 * 1024), (63 * 1024 + 5, 64 * 1024), (64 * 1024, 64 * 1024),
                                        (64 * 1024, 64 * 1024 + 1), (1, 60_000)])
def test_gpu_sort_few_tiles(live, bound, n_cells):
    edges.test_gpu_sort_edges(4, live, bound, n_cells)
