"""Nearest-seed labels of grids with few cells in each brick of 8 x 8 x 32, which go by tiles of cells in linear order: flat along
each axis, rows that end within a tile, seeds few and in several chunks, 64-bit keys.  Equal to the oracle's."""
import time

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
EUC, MAN, CHE = 0, 1, 2
# 8192 and 8064 bricks (the line is between), 8320, and 8192 flat along x and y
DIMS = [(1024, 512, 1), (1024, 504, 1), (1037, 507, 3), (1, 2047, 1021), (1021, 1, 2048)]


def random_seeds(grid, n, seed):
    at = np.argwhere(grid)
    at = at[np.sort(np.random.default_rng(seed).choice(len(at), n, replace=False))]
    return np.concatenate([at, np.arange(n)[:, None] + 2], 1).astype(np.uint32)


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("dist", [EUC, MAN, CHE])
def test_thin_grids(vf, dims, dist):
    grid = (np.random.default_rng(dims[0]).random(dims) < 0.02).astype(np.uint16)
    grid[-1, -1, -1] = 1
    with vf.Grid(dims, *BOX) as g:
        for n in (1, 16, 17, 200, 1030):
            print("naive", dims, dist, n, flush=True)
            seeds = random_seeds(grid, n, n)
            g.write(grid)
            g.fracture_naive(seeds, dist)
            np.testing.assert_array_equal(g.read(), O.naive(grid, seeds, dist))


def test_a_flat_grid_takes_no_bricks(vf):
    dims = (2048, 2048, 1)
    grid = (np.random.default_rng(0).random(dims) < 0.05).astype(np.uint16)
    seeds = random_seeds(grid, 32, 1)
    took = []
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        for _ in range(6):
            t0 = time.perf_counter()
            g.fracture_naive(seeds, EUC)
            took.append(time.perf_counter() - t0)
        np.testing.assert_array_equal(g.read(), O.naive(grid, seeds, EUC))
    print("naive labels of a flat grid:", min(took), flush=True)
    assert min(took) < 150e-6  # 272 us by bricks, 54 by tiles
