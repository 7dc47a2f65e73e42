"""Voxelization where a wave's pairs belong to one, two, three or more triangles, which change their occupancy words alone or
together, and whose columns have one, two or more cells: triangles that cover many columns of flat grids, slivers a few
columns wide among them, and two meshes in a batch.  Occupancy equals the oracle's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.0, -1.0, -1.0], [1.0, 1.0, 1.0])


def sheet(seed, n, wide, thin):
    """n large triangles, each followed by a few thin ones across it: waves of every number of triangles."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        out.append(rng.uniform(-1, 1, 3) * [0.3, 0.3, 0.9] + rng.uniform(-wide, wide, (3, 3)) * [1, 1, 0.5])
        for _ in range(int(rng.integers(0, 6))):
            a = rng.uniform(-0.9, 0.9, 3)
            out.append(a + np.array([[0, 0, 0], [thin, 0, rng.uniform(-0.2, 0.2)], [0, rng.uniform(0.1, 0.9), 0]]))
    v = np.array(out, np.float32)
    return v.reshape(-1, 3), np.arange(3 * len(v), dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("dims", [(200, 190, 1), (150, 140, 2), (90, 100, 3), (120, 60, 16), (64, 70, 40)])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 30])
def test_waves_of_few_triangles(vf, dims, n):
    for thin in (0.02, 0.1):
        print("sheet", dims, n, thin, flush=True)
        xyz, tri = sheet(n, n, 0.9, thin)
        with vf.Grid(dims, *BOX) as g:
            g.voxelize(xyz, tri)
            np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, *BOX, dims))


def test_waves_of_two_grids(vf):
    meshes = [sheet(s, 4, 0.7, 0.05) for s in (8, 9)]
    dims = [(70, 60, 5), (50, 80, 2)]
    jobs, outs = [], []
    for (xyz, tri), d in zip(meshes, dims):
        j = vf.make_job(xyz, tri, d, *BOX, 1, 5, vf.NAIVE, vf.EUCLIDEAN)
        j.boundary_size = 0
        out = np.zeros(d, np.uint16)
        j.labels_out = out.ctypes.data
        jobs.append(j)
        outs.append(out)
    with vf.Batch() as b:
        assert [r["status"] for r in b.run(jobs)] == [0, 0]
    for (xyz, tri), d, out in zip(meshes, dims, outs):
        np.testing.assert_array_equal(out != 0, O.voxelize(xyz, tri, *BOX, d) != 0)


def test_columns_far_outside_an_axis(vf):
    # steep slivers beside columns of many cells: an axis excludes the whole column by quotients far below or above any
    # cell's number, which are clamped before they become integers
    rng = np.random.default_rng(3)
    n = 400
    a = rng.uniform(-0.9, 0.9, (n, 1, 3))
    v = a + rng.uniform(-1, 1, (n, 3, 3)) * np.array([0.6, 0.6, 1e-6])
    v[::2, 2] = v[::2, 1] + [1e-7, 0.4, 1e-7]
    v[::3, :, 2] += rng.uniform(-0.5, 0.5, (len(v[::3]), 3))
    xyz, tri = v.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    for dims in ((40, 50, 64), (30, 30, 200), (300, 20, 33)):
        with vf.Grid(dims, *BOX) as g:
            g.voxelize(xyz, tri)
            np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, *BOX, dims))
