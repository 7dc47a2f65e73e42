"""Marching cubes on grids whose columns are shorter than, as long as and longer than a unit of 8 points, whose rows are
aligned to nothing, with flagged, FREE and top labels, one label wanted or all.  Meshes equal the oracle's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
DIMS = [(1, 1, 1), (3, 4, 5), (9, 5, 7), (6, 6, 8), (5, 7, 9), (4, 9, 15), (3, 8, 16), (7, 8, 23), (10, 3, 65), (24, 25, 26)]


def cases(dims):
    rng = np.random.default_rng(sum(dims))
    few = rng.integers(0, 4, dims, np.uint16)  # EMPTY, FREE and two labels, mixed at every point
    yield "few", few
    many = rng.integers(0, 40, dims, np.uint16)
    many[rng.random(dims) < 0.5] = 0
    many[(rng.random(dims) < 0.3) & (many > 1)] |= 0x8000
    yield "many", many
    blocks = np.full(dims, 5, np.uint16)
    blocks[:, :, dims[2] // 2:] = 9
    blocks[dims[0] // 2:] = 0
    yield "blocks", blocks
    top = np.where(rng.random(dims) < 0.5, 0x7FFE, 2).astype(np.uint16)
    top[rng.random(dims) < 0.1] |= 0x8000
    yield "top", top
    odd = few.copy()
    odd[rng.random(dims) < 0.1] = 0x8000  # a flagged EMPTY cell
    yield "flagged empty", odd
    yield "solid", np.full(dims, 0x8003, np.uint16)


@pytest.mark.parametrize("dims", DIMS)
def test_units(vf, dims):
    with vf.Grid(dims, *BOX) as g:
        for name, grid in cases(dims):
            print("marching cubes", dims, name, flush=True)
            g.write(grid)
            for label in (vf.ALL_LABELS, 3):
                got, want = g.marching_cubes(label), O.marching_cubes(grid, *BOX, label)
                for k in ("labels", "voff", "toff", "tri", "flag", "xyz"):
                    np.testing.assert_array_equal(got[k], want[k], err_msg="%s %s" % (name, k))
