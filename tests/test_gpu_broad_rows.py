"""Broad phase in crowded scenes: rows of cells shorter and longer than the
candidates in flight, waves whose objects share their cells and waves whose
objects do not, against the oracle, and what a crowded scene takes."""
import time

import numpy as np
import pytest

import ogjk
from ogjk import gen
from test_gpu_broad import check_equal, torch_cuda  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cell", [(7, 8, 9), (15, 16, 17), (1, 3, 24, 64), (65, 150, 2)])
@pytest.mark.parametrize("grid_size", [3, 5])
def test_row_lengths(torch_cuda, per_cell, grid_size):  # noqa: F811
    half = 5.0
    edge = 2.0 * half / grid_size
    rng = np.random.default_rng(sum(per_cell) + grid_size)
    rows = []
    for c in np.ndindex(grid_size, grid_size, grid_size):
        if rng.random() < 0.3:
            continue  # empty cells and rows between
        m = int(rng.choice(per_cell))
        centre = (np.array(c) + 0.5) * edge - half
        rows.append(np.concatenate([centre + rng.uniform(-0.45 * edge, 0.45 * edge, (m, 3)),
                                    rng.uniform(0.05, 0.5 * edge, (m, 1))], 1))
    s = rng.permutation(np.concatenate(rows).astype(np.float32))
    grid = ogjk.Grid(edge, half, grid_size, 0)
    found = check_equal(torch_cuda, f"rows {per_cell} in {grid_size}^3", s, grid)
    assert found > 0


def test_crowded_scene_is_walked_by_rows(torch_cuda):  # noqa: F811
    """10,000 spheres at 150 a cell: three cells of a row at once, so well under
    the time of the capped form, which takes them one by one (0.64 of it; 0.83
    while every index waited for its sphere)."""
    torch = torch_cuda
    n, half, g = 10_000, 4.6, 4
    x = torch.from_numpy(gen.spheres(n, seed=1, box=half, rmin=0.2, rmax=1.0)).cuda()

    def seconds(cap):
        bp = ogjk.BroadPhase(n, ogjk.Grid(2 * half / g, half, g, cap), max_pairs=50 * n)
        pairs, found = bp(x)
        best = 1e9
        for _ in range(6):
            t = time.perf_counter()
            for _ in range(5):
                bp(x)
            best = min(best, time.perf_counter() - t)
        return best, found

    (rows, f0), (cells, f1) = seconds(0), seconds(4096)
    print(f"\nby rows {rows / 5 * 1e6:.0f} us, by cells {cells / 5 * 1e6:.0f} us", flush=True)
    assert f0 == f1 > n
    assert rows < 0.75 * cells
