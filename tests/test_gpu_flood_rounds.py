"""Flood rounds whose worklists are shorter than, about as long as and longer than the workgroups that serve
them, on solid boxes, where the flood without noise is the nearest seed in the 6- or 26-neighbour distance
(ties to the first seed), alone and several to a table."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
EUC, MAN, CHE = 0, 1, 2


def nearest(dims, seeds, dist):
    ax = [np.arange(n, dtype=np.int32) for n in dims]
    best = np.full(dims, 1 << 20, np.int32)
    label = np.zeros(dims, np.uint16)
    for x, y, z, w in seeds.astype(np.int64):
        d = [np.abs(a - c).reshape([-1 if k == i else 1 for k in range(3)]) for i, (a, c) in enumerate(zip(ax, (x, y, z)))]
        t = d[0] + d[1] + d[2] if dist == MAN else np.maximum(np.maximum(d[0], d[1]), d[2])
        label = np.where(t < best, np.uint16(w), label)
        best = np.minimum(best, t)
    return label


def draw_seeds(dims, n, seed):
    rng = np.random.default_rng(seed)
    cells = rng.choice(dims[0] * dims[1] * dims[2], n, replace=False)
    s = np.stack(np.unravel_index(np.sort(cells), dims) + (np.arange(n) + 2,), 1)
    return s.astype(np.uint32)


@pytest.mark.parametrize("dims,n,dist", [((9, 3, 5), 1, MAN), ((33, 57, 70), 3, CHE), ((64, 8, 200), 5, MAN),
                                         ((136, 152, 144), 200, CHE), ((256, 248, 240), 3, MAN), ((250, 241, 243), 2, CHE)])
def test_solid_box_is_nearest_seed(vf, dims, n, dist):
    print("flood of a solid box", dims, n, dist, flush=True)
    seeds = draw_seeds(dims, n, sum(dims))
    with vf.Grid(dims, *BOX) as g:
        g.write(np.ones(dims, np.uint16))
        for _ in range(2):  # a second growth of the same grid
            g.fracture_flood(seeds, dist)
            np.testing.assert_array_equal(g.read(), nearest(dims, seeds, dist))


def test_tables_of_uneven_jobs_count_their_work(vf):
    # jobs of few and many bricks share each round's lists; every brick with cells is visited, each visit
    # sweeps at least once, and the counts of a table sum to those jobs' own work
    xyz, tri = vf.vessel_mesh(11, *vf.vessel_segments(6000))
    dev = vf.DeviceMesh(xyz, tri)
    edges = (16, 200, 24, 64, 128, 20)
    jobs = [dev.job((e, e, e), *BOX, 4, 9 + e, 1, (EUC, MAN, CHE)[i % 3], noise_seed=e, noise_amp=i % 3)
            for i, e in enumerate(edges)]
    alone = [vf.plain_run([j])[0] for j in jobs]
    with vf.Batch() as b:
        for _ in range(3):
            res = b.run(jobs)
            for e, r, a in zip(edges, res, alone):
                print("table", e, r["flood_bricks"], r["flood_sweeps"], flush=True)
                assert r["status"] == 0 and r["checksum"] == a["checksum"] and r["occupied"] == a["occupied"]
                assert r["flood_bricks"] >= r["occupied"] / 512 and r["flood_sweeps"] >= r["flood_bricks"]
                assert r["flood_levels"] > 0
    dev.close()
