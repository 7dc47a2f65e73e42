"""Stages that go by the occupancy words (32 cells of a column each) and by bricks of 8 x 8 x 32 cells, on grids whose
edges fall on, before and after word and brick ends: occupancy, seed candidates, both fractures, and voxelizing into a
grid that holds labels.  Integer results equal the oracle's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
EUC, MAN, CHE = 0, 1, 2
DIMS = [(3, 4, 1), (9, 11, 31), (8, 8, 32), (10, 7, 33), (17, 5, 64), (6, 9, 65), (5, 16, 130), (40, 33, 100)]


def random_grid(dims, density=0.6):
    rng = np.random.default_rng(sum(dims))
    g = (rng.random(dims) < density).astype(np.uint16)
    g[tuple(slice(1, n - 1) for n in dims)] |= rng.random(tuple(max(0, n - 2) for n in dims)) < 0.9  # some inner cells
    return g


def random_seeds(grid, n, seed):
    rng = np.random.default_rng(seed)
    at = np.argwhere(grid)
    at = at[np.sort(rng.choice(len(at), min(n, len(at)), replace=False))]
    return np.concatenate([at, np.arange(len(at))[:, None] + 2], 1).astype(np.uint32)


@pytest.mark.parametrize("dims", DIMS)
def test_occupancy_and_seed_candidates(vf, dims):
    print("occupancy", dims, flush=True)
    grid = random_grid(dims)
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        np.testing.assert_array_equal(g.occupancy(), grid.astype(np.uint8))
        assert g.count_occupied() == int(grid.sum())
        for location in (vf.SEED_INNER, vf.SEED_OUTER, vf.SEED_BOTH):
            for n in (1, 3, 40):
                try:
                    want = O.seed_uniform(grid, n, 5 + n, location)
                except Exception:
                    want = None
                if want is None:
                    with pytest.raises(vf.VfError):
                        g.seed_uniform(n, 5 + n, location)
                else:
                    np.testing.assert_array_equal(g.seed_uniform(n, 5 + n, location), want)


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("dist", [EUC, MAN, CHE])
def test_fractures_on_odd_edges(vf, dims, dist):
    print("fractures", dims, dist, flush=True)
    grid = random_grid(dims)
    with vf.Grid(dims, *BOX) as g:
        for n in (2, 16, 17, 300):  # all seeds applied to every cell, or the far ones dropped by brick
            seeds = random_seeds(grid, n, n)
            g.write(grid)
            g.fracture_naive(seeds, dist)
            np.testing.assert_array_equal(g.read(), O.naive(grid, seeds, dist))
        seeds = random_seeds(grid, 20, 3)
        g.write(grid)
        g.fracture_flood(seeds, dist, noise_seed=4, noise_amp=2)
        np.testing.assert_array_equal(g.read(), O.flood(grid, seeds, 6 if dist == MAN else 26, 4, 2))


@pytest.mark.parametrize("dims,n,dist", [((24, 31, 70), 1024, EUC), ((24, 31, 70), 1025, MAN), ((24, 31, 70), 2600, CHE),
                                         ((2000, 3, 40), 40, EUC), ((2047, 9, 5), 33, EUC)])
def test_naive_seed_chunks_and_wide_keys(vf, dims, n, dist):
    # several chunks of seeds, and grids whose Euclidean keys need 64 bits or rank by float roots
    print("naive", dims, n, dist, flush=True)
    grid = random_grid(dims)
    seeds = random_seeds(grid, n, 9)
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        g.fracture_naive(seeds, dist)
        np.testing.assert_array_equal(g.read(), O.naive(grid, seeds, dist))


@pytest.mark.parametrize("dims", [(40, 36, 31), (33, 40, 65)])
def test_voxelize_into_labels(vf, dims):
    # RegularGrid::fill only sets cells: the others keep their labels
    a, b = (vf.vessel_mesh(s, *vf.vessel_segments(3000)) for s in (1, 2))
    occ_a, occ_b = (O.voxelize(*m, *BOX, dims) for m in (a, b))
    with vf.Grid(dims, *BOX) as g:
        g.voxelize(*a)
        seeds = g.seed_uniform(6, 3)
        g.fracture_naive(seeds, EUC)
        lab = g.read()
        np.testing.assert_array_equal(lab, O.naive(O.occ_to_grid(occ_a), seeds, EUC))
        g.voxelize(*b)
        np.testing.assert_array_equal(g.read(), np.where(occ_b != 0, np.uint16(1), lab))
        np.testing.assert_array_equal(g.occupancy(), ((occ_a | occ_b) != 0).astype(np.uint8))
        g.set_aabb(*BOX, dims)
        assert not g.read().any() and not g.occupancy().any() and g.count_occupied() == 0


def test_small_and_large_jobs_share_a_table(vf):
    # bricks and word tiles of uneven jobs, seeded anywhere, outside and inside, in one table
    xyz, tri = vf.vessel_mesh(5, *vf.vessel_segments(9000))
    dev = vf.DeviceMesh(xyz, tri)
    edges = [(20, 20, 20), (61, 45, 33), (96, 96, 96), (31, 64, 130)]
    jobs, out = [], []
    for i, e in enumerate(edges * 2):
        j = dev.job(e, *BOX, 3 + 9 * i, 7 + i, i // len(edges), (EUC, MAN, CHE)[i % 3], noise_seed=i, noise_amp=2,
                    seed_location=(vf.SEED_BOTH, vf.SEED_OUTER)[i % 2])
        lab = np.empty(e, np.uint16)
        j.labels_out = lab.ctypes.data
        jobs.append(j)
        out.append(lab)
    with vf.Batch() as b:
        for _ in range(2):
            res = b.run(jobs)
            for i, (j, lab, r) in enumerate(zip(jobs, out, res)):
                e = edges[i % len(edges)]
                occ = O.occ_to_grid(O.voxelize(xyz, tri, *BOX, e))
                seeds = O.seed_uniform(occ, j.num_seeds, j.seed, j.seed_location)
                ref = O.naive(occ, seeds, j.distance) if j.algorithm == 0 else \
                    O.flood(occ, seeds, 6 if j.distance == MAN else 26, j.noise_seed, 2)
                ref = O.detect_boundaries(ref, 1)
                assert r["status"] == 0 and r["occupied"] == int((occ != 0).sum())
                np.testing.assert_array_equal(lab, ref, err_msg=str((i, e)))
                assert r["checksum"] == O.checksum(ref)
    dev.close()
