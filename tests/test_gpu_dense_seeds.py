"""Uniform seed draws that take nearly every candidate: the last cells take about as many draws each as there are
candidates.  Equal to the oracle's draws, which go one by one."""
import time

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
DIMS = (32, 30, 40)


@pytest.mark.parametrize("cells,seeds", [(1, 1), (2, 2), (64, 64), (255, 255), (256, 256), (257, 257), (300, 257), (1000, 999),
                                         (2048, 2000), (4096, 4096), (4200, 4096), (20000, 4096)])
def test_draws_of_nearly_every_cell(vf, cells, seeds):
    print("draw", seeds, "of", cells, flush=True)
    grid = np.zeros(DIMS, np.uint16)
    grid.ravel()[np.random.default_rng(cells).choice(grid.size, cells, replace=False)] = 1
    with vf.Grid(DIMS, *BOX) as g:
        g.write(grid)
        for key in (1, 2):
            t0 = time.perf_counter()
            got = g.seed_uniform(seeds, key)
            took = time.perf_counter() - t0
            np.testing.assert_array_equal(got, O.seed_uniform(grid, seeds, key))
            assert took < 0.4  # 1.37 s with a draw a step for the last cell; 16 ms
