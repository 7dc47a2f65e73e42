"""Conversions between labels, occupancy words and occupancy bytes, which take 8 cells of a column at a time: columns shorter
than that, of whole groups and words and a few cells more or less, and more groups than one step has threads."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
DIMS = [(70, 60, n) for n in (1, 2, 7, 8, 9, 15, 16, 17, 24, 25, 31, 32, 33, 40, 41, 63, 64, 65, 95, 97, 129)] + [(1, 1, 1), (1, 3, 13), (2048, 1900, 2), (401, 330, 223)]


@pytest.mark.parametrize("dims", DIMS)
def test_labels_and_occupancy(vf, dims):
    print("columns", dims, flush=True)
    rng = np.random.default_rng(dims[2])
    dense = np.ones(dims, np.uint16)
    sparse = np.where(rng.random(dims) < 0.3, rng.integers(1, 1 << 16, dims), 0).astype(np.uint16)
    sparse[0, 0, -1] = 0x8000  # flagged, and not EMPTY
    xyz, tri = vf.vessel_mesh(5, *vf.vessel_segments(3000))
    with vf.Grid(dims, *BOX) as g:
        for grid in (dense, sparse, dense):  # no bits of the grid before are left
            g.write(grid)
            np.testing.assert_array_equal(g.occupancy(), (grid != 0).astype(np.uint8))
            assert g.count_occupied() == int((grid != 0).sum())
            np.testing.assert_array_equal(g.read(), grid)
        g.write(sparse)
        occ = (sparse != 0).astype(np.uint16)
        n = min(9, int(occ.sum()))
        np.testing.assert_array_equal(g.seed_uniform(n, 4), O.seed_uniform(occ, n, 4))
        want = O.voxelize(xyz, tri, *BOX, dims)
        g.voxelize(xyz, tri)  # into a grid that holds labels
        merged = np.where(want != 0, 1, sparse).astype(np.uint16)
        np.testing.assert_array_equal(g.read(), merged)
        np.testing.assert_array_equal(g.occupancy(), (merged != 0).astype(np.uint8))
        g.set_aabb(*BOX, dims)
        g.voxelize(xyz, tri)
        np.testing.assert_array_equal(g.occupancy(), (want != 0).astype(np.uint8))
        np.testing.assert_array_equal(g.read(), want)
