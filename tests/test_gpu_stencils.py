"""Erosion and isolated cells on grids whose edges fall on, before and after the bricks of 8 x 8 x 32 cells, with windows
of every side, on labels with and without the boundary bit, FREE and EMPTY cells.  Cells equal the oracle's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
DIMS = [(1, 1, 1), (3, 5, 1), (8, 8, 32), (9, 7, 33), (16, 17, 31), (25, 8, 70)]


def labelled(dims, seed):
    rng = np.random.default_rng(seed)
    g = np.repeat(np.repeat(np.repeat(rng.integers(0, 5, [-(-n // 5) for n in dims]), 5, 0), 5, 1), 5, 2)
    g = g[:dims[0], :dims[1], :dims[2]].astype(np.uint16)  # pieces of 5 cells, some EMPTY and FREE
    stray = rng.random(dims) < 0.1
    g[stray] = rng.integers(0, 300, int(stray.sum()))
    g[rng.random(dims) < 0.15] |= 0x8000
    g[g == 0x8000] = 0
    return g


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("kind,size", [(0, 1), (0, 3), (1, 3), (2, 3), (2, 4), (0, 5), (1, 7), (2, 9), (2, 15)])
def test_windows(vf, dims, kind, size):
    print("erode", dims, kind, size, flush=True)
    grid = labelled(dims, sum(dims) + size)
    with vf.Grid(dims, *BOX) as g:
        for iters, prob, thr in ((1, 1.0, 0.6), (2, 0.5, 0.9), (0, 0.5, 0.5)):
            g.write(grid)
            g.erode(kind, size, iters, prob, thr, 77)
            want = O.erode(grid.copy(), kind, size, iters, prob, thr, 77)
            np.testing.assert_array_equal(g.read(), want)
            assert g.count_occupied() == int((want != 0).sum())


@pytest.mark.parametrize("dims", DIMS)
def test_isolated_cells(vf, dims):
    grid = labelled(dims, sum(dims))
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        g.remove_isolated_cells()
        np.testing.assert_array_equal(g.read(), O.remove_isolated_cells(grid))
