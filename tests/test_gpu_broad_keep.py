"""The broad phase where an object's partners just fit, or do not, what the
count pass keeps of them, in cells of up to the largest rank-scanned occupancy,
at corners, edges and the middle of the grid and with empty rows between."""
import numpy as np
import pytest

import ogjk
from test_gpu_broad import check_equal, torch_cuda  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid_size", [1, 2, 3, 9])
@pytest.mark.parametrize("counts", [(1,), (16, 17), (17, 18, 33), (1, 2, 15, 16, 17, 64)])
def test_kept_partners(torch_cuda, grid_size, counts):  # noqa: F811
    half = 9.0
    edge = 2.0 * half / grid_size
    rng = np.random.default_rng(len(counts) * 10 + grid_size)
    cells = [(0, 0, 0), (grid_size - 1,) * 3, (grid_size // 2, 0, grid_size - 1),
             (grid_size // 2,) * 3, (0, grid_size - 1, grid_size // 2), (grid_size - 1, 0, 0)]
    rows = []
    for m, c in zip(counts, cells):
        centre = (np.array(c) + 0.5) * edge - half
        rows.append(np.concatenate([centre + rng.uniform(-0.05, 0.05, (m, 3)),
                                    np.full((m, 1), 0.5)], 1))
    s = rng.permutation(np.concatenate(rows).astype(np.float32))
    grid = ogjk.Grid(edge, half, grid_size, 0)
    found = check_equal(torch_cuda, f"keep {counts} in {grid_size}^3", s, grid)
    assert grid_size < 3 or found >= sum(m * (m - 1) // 2 for m in counts)
    check_equal(torch_cuda, "cut short", s, grid, max_pairs=max(found // 2, 1))
