"""Single-grid calls whose small inputs and results travel with the launches: seed lists around one launch's worth, a
cleared box read by every stage that can come first, counts of small and large labels, triangle counts around the
one-launch scan, floods that keep going after their first drain.  Integer results equal the oracle's or numpy's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
EUC, MAN, CHE = 0, 1, 2


@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 5, 7), (16, 16, 33), (40, 24, 50), (130, 90, 64)])
@pytest.mark.parametrize("labels", [[1, 2], [2, 1023], [1023, 1024], [0x7FFF, 5, 1025], list(range(2, 3000))])
def test_histogram(vf, dims, labels):
    print("histogram", dims, labels[:4], flush=True)
    rng = np.random.default_rng(dims[0] + len(labels))
    g = rng.choice(np.array(labels, np.uint16), dims)
    g[rng.random(dims) < 0.4] = 0
    g[rng.random(dims) < 0.2] |= 0x8000  # boundary cells count with their label
    want = np.bincount((g & 0x7FFF)[g > 1].ravel(), minlength=65536).astype(np.uint32)
    with vf.Grid(dims, *BOX) as grid:
        grid.write(g)
        for n in (65536, 1, 2, 700, 1024, 1025, 40000, 65536):  # no counts left over from the call before
            np.testing.assert_array_equal(grid.histogram(n), want[:n])


@pytest.mark.parametrize("n", [127, 128, 129, 300, 1023, 1025])
def test_seed_lists(vf, n):
    dims = (18, 17, 40)
    rng = np.random.default_rng(n)
    grid = (rng.random(dims) < 0.8).astype(np.uint16)
    at = np.argwhere(grid)[rng.choice(int(grid.sum()), n, replace=False)]
    seeds = np.concatenate([at, np.arange(n)[:, None] + 2], 1).astype(np.uint32)
    with vf.Grid(dims, *BOX) as g:
        for dist in (MAN, CHE):
            g.write(grid)
            g.fracture_naive(seeds, dist)
            np.testing.assert_array_equal(g.read(), O.naive(grid, seeds, dist))
            seeds[:, 3] = 2 + seeds[:, 3] % 254  # flood regions have 8-bit ids
            g.write(grid)
            g.fracture_flood(seeds, dist)
            np.testing.assert_array_equal(g.read(), O.flood(grid, seeds, 6 if dist == MAN else 26))


def test_a_new_box_is_empty_to_every_stage(vf):
    dims = (20, 21, 45)
    xyz, tri = vf.vessel_mesh(5, *vf.vessel_segments(3000))
    first = [lambda g: np.testing.assert_array_equal(g.read(), np.zeros(dims, np.uint16)),
             lambda g: np.testing.assert_array_equal(g.occupancy(), np.zeros(dims, np.uint8)),
             lambda g: np.testing.assert_array_equal(g.histogram(), np.zeros(65536, np.uint32)),
             lambda g: g.detect_boundaries(1),
             lambda g: g.undo_mask(),
             lambda g: g.homogenize(),
             lambda g: None]
    with vf.Grid(dims, *BOX) as g:
        for k, stage in enumerate(first):
            print("first stage", k, flush=True)
            g.voxelize(xyz, tri)
            assert g.count_occupied() > 0
            g.set_aabb(*BOX, dims)
            stage(g)
            assert g.count_occupied() == 0
            with pytest.raises(vf.VfError):
                g.seed_uniform(2, 1)
            np.testing.assert_array_equal(g.read(), np.zeros(dims, np.uint16))


@pytest.mark.parametrize("nt", [1, 4095, 4096, 4097, 8191, 8192, 8193])  # two counts a triangle: scans around 8192 and 16384
def test_triangle_counts(vf, nt):
    print("triangles", nt, flush=True)
    dims = (30, 33, 36)
    rng = np.random.default_rng(nt)
    v = (rng.uniform(-1, 1, (nt, 1, 3)) + rng.uniform(-0.12, 0.12, (nt, 3, 3))).astype(np.float32)
    xyz, tri = v.reshape(-1, 3), np.arange(3 * nt, dtype=np.uint32).reshape(-1, 3)
    with vf.Grid(dims, *BOX) as g:
        g.voxelize(xyz, tri)
        np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, *BOX, dims))
        if nt > 1:
            tri[nt // 2, 1] = 3 * nt  # one bad index is still found, and the grid still usable
            with pytest.raises(vf.VfError):
                g.voxelize(xyz, tri)
            tri[nt // 2, 1] = 0
            g.set_aabb(*BOX, dims)
            g.voxelize(xyz, tri)
            np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, *BOX, dims))


@pytest.mark.parametrize("dist", [MAN, CHE])
def test_long_floods(vf, dist):
    # a corridor that winds through the grid: one brick a round, many more rounds than are queued ahead
    dims = (41, 40, 40)
    grid = np.zeros(dims, np.uint16)
    grid[::4, :, :] = 1
    for k, x in enumerate(range(2, 40, 4)):
        grid[x - 2:x + 3, 0 if k % 2 else -1, :] = 1
    grid[:, :, 8:24] = 0
    grid[0, 3, 8:24] = 1
    seeds = np.array([[0, 0, 0, 2], [20, 20, 39, 3]], np.uint32)
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        g.fracture_flood(seeds, dist, noise_seed=3, noise_amp=1)
        np.testing.assert_array_equal(g.read(), O.flood(grid, seeds, 6 if dist == MAN else 26, 3, 1))
