"""The voxelizer's shared pair lists: triangles of every extent around the word (32 cells of a column), list and wave
ends, words that many triangles of a wave change at once, waves that span two jobs, and coordinates so large that the
cell test's arithmetic overflows.  Occupancy equals the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.0, -1.0, -1.0], [1.0, 1.0, 1.0])


def soup(seed, n, size, huge=0.0):
    """n triangles of about `size`, some repeated, flat, along an axis or (huge) with far vertices."""
    rng = np.random.default_rng(seed)
    v = rng.uniform(-1.1, 1.1, (n, 1, 3)) + rng.uniform(-size, size, (n, 3, 3))
    kind = rng.integers(0, 8, n)
    v[kind == 0, 1] = v[kind == 0, 0]  # two equal vertices
    v[kind == 1, :, 2] = v[kind == 1, :1, 2]  # flat in z
    v[kind == 2, :, 0] = v[kind == 2, :1, 0]  # and in x
    v[kind == 3] = np.round(v[kind == 3] * 8) / 8  # vertices on cell faces
    if huge:
        far = rng.random((n, 3)) < 0.4
        v[far] *= huge
    v = np.concatenate([v, v[: n // 3], v[: n // 5]]).astype(np.float32)  # the same words, toggled two and three times
    return v.reshape(-1, 3), np.arange(3 * len(v), dtype=np.uint32).reshape(-1, 3)


def check(vf, dims, xyz, tri):
    with vf.Grid(dims, *BOX) as g:
        g.voxelize(xyz, tri)
        np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, *BOX, dims))


@pytest.mark.parametrize("dims", [(5, 7, 1), (16, 16, 16), (9, 12, 31), (8, 24, 33), (20, 3, 64), (31, 17, 100)])
@pytest.mark.parametrize("n,size", [(1, 0.9), (7, 0.5), (63, 0.3), (400, 0.08), (150, 1.5)])
def test_triangles_of_every_extent(vf, dims, n, size):
    print("soup", dims, n, size, flush=True)
    check(vf, dims, *soup(n + sum(dims), n, size))


@pytest.mark.parametrize("huge", [9e11, 1.1e12, 1e19, 1e25, 2e38])
def test_far_vertices(vf, huge):
    print("far", huge, flush=True)
    check(vf, (12, 18, 40), *soup(5, 60, 0.4, huge))


def test_far_grid(vf):
    lo, hi, dims = [-3e12] * 3, [3e12] * 3, (9, 10, 35)
    xyz, tri = soup(6, 80, 0.4)
    xyz = xyz * np.float32(3e12)
    with vf.Grid(dims, lo, hi) as g:
        g.voxelize(xyz, tri)
        np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, lo, hi, dims))


@pytest.mark.parametrize("offset", [0.0, 1.0, 100.0, 1e4, 3e6])
@pytest.mark.parametrize("dims", [(12, 18, 40), (40, 40, 33)])
def test_grids_away_from_the_origin(vf, offset, dims):
    # the further away, the coarser a cell's planes and offsets round, and the more cells lie too near an interval's end
    print("offset", offset, dims, flush=True)
    lo, hi = [offset - 1.0, 2 * offset - 1.0, 1.0 - offset], [offset + 1.0, 2 * offset + 1.0, 3.0 - offset]
    xyz, tri = soup(int(offset) % 97 + dims[0], 250, 0.25)
    xyz = (xyz + (np.array(lo) + np.array(hi)) / 2).astype(np.float32)
    with vf.Grid(dims, lo, hi) as g:
        g.voxelize(xyz, tri)
        np.testing.assert_array_equal(g.read(), O.voxelize(xyz, tri, lo, hi, dims))


@pytest.mark.parametrize("seed", range(6))
def test_slivers_and_aligned_edges(vf, seed):
    rng = np.random.default_rng(seed)
    n, dims = 300, (33, 31, 64)
    v = rng.uniform(-0.9, 0.9, (n, 1, 3)) + rng.uniform(-0.3, 0.3, (n, 3, 3)) * 10.0 ** rng.uniform(-6, 0, (n, 1, 3))
    kind = rng.integers(0, 5, n)
    v[kind == 1, 1] = v[kind == 1, 0] + np.array([0.3, 0, 0])  # an edge along each coordinate
    v[kind == 2, 1] = v[kind == 2, 0] + np.array([0, 0.3, 0])
    v[kind == 3, 1] = v[kind == 3, 0] + np.array([0, 0, 0.3])
    v[kind == 4] = np.round(v[kind == 4] * 16) / 16  # corners of cells and of boxes
    xyz = v.reshape(-1, 3).astype(np.float32)
    check(vf, dims, xyz, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))


def test_jobs_share_waves(vf):
    dims = [(6, 5, 40), (16, 16, 16), (3, 3, 3), (20, 9, 70), (8, 8, 8)]
    meshes = [soup(20 + i, 3 + 2 * i, 0.6) for i in range(len(dims))]
    out = [np.zeros(d, np.uint16) for d in dims]
    ref = [O.voxelize(*m, *BOX, d) for m, d in zip(meshes, dims)]
    keep, jobs = [], []
    for d, m, o in zip(dims, meshes, out):
        jobs.append(vf.make_job(*m, d, *BOX, 1, 1, vf.NAIVE, vf.EUCLIDEAN, keep=keep))
        jobs[-1].labels_out = o.ctypes.data
    for r in vf.Batch(graphs=False).run(jobs):
        assert r["status"] == 0
    for o, r in zip(out, ref):
        np.testing.assert_array_equal(o & 0x7FFF != 0, r != 0)
