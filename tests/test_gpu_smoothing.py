"""Smoothing step counts: none, one or several of either kind, a second smoothing of the same mesh, and grids of one
launch that stop at different steps.  Positions equal the oracle's, bit for bit (sums are in integers)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])


def fractured(vf, dims, n, seed):
    xyz, tri = vf.vessel_mesh(seed, *vf.vessel_segments(6000))
    g = vf.Grid(dims, *BOX)
    g.voxelize(xyz, tri)
    g.fracture_naive(g.seed_uniform(n, seed), 0)
    g.detect_boundaries(1)
    return g


@pytest.mark.parametrize("sm", [(0, 0.5, 0, 0.5), (1, 0.9, 0, 0.2), (0, 0.9, 1, 0.2), (2, 1.0, 3, 0.0), (3, 0.3, 2, 1.0), (5, 0.9, 1, 0.4)])
def test_step_counts(vf, sm):
    print("smooth", sm, flush=True)
    with fractured(vf, (40, 37, 45), 9, 4) as g:
        r = O.marching_cubes(g.read(), *BOX, smooth=sm)
        g.marching_cubes()
        g.smooth_mesh(*sm)
        np.testing.assert_array_equal(g.read_mesh()["xyz"], r["xyz"])


def test_scattered_cells(vf):
    # many one-cell pieces: vertices of few triangles, all or no triangles flagged
    dims = (12, 13, 14)
    rng = np.random.default_rng(6)
    grid = rng.integers(0, 9, dims, np.uint16)
    grid[rng.random(dims) < 0.3] |= 0x8000
    grid[(grid & 0x7FFF) < 2] = 0
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        for sm in ((2, 0.7, 2, 0.3), (1, 0.5, 4, 0.5)):
            g.marching_cubes()
            g.smooth_mesh(*sm)
            np.testing.assert_array_equal(g.read_mesh()["xyz"], O.marching_cubes(grid, *BOX, smooth=sm)["xyz"])


def test_grids_of_one_launch_stop_at_different_steps(vf):
    xyz, tri = vf.vessel_mesh(8, *vf.vessel_segments(6000))
    dev = vf.DeviceMesh(xyz, tri)
    steps = [(0, 0.9, 0, 0.2), (3, 0.9, 1, 0.2), (1, 0.4, 5, 0.6), (4, 0.8, 0, 0.2), (0, 0.9, 2, 0.3)]
    edges = (24, 40, 33, 48, 28)

    def run(which):
        jobs, bufs = [], []
        for i in which:
            e = (edges[i],) * 3
            j = dev.job(e, *BOX, 5 + i, 30 + i, 1, 0, marching_cubes=1, smooth=steps[i])
            b = vf.MeshBuffers(200000, 400000)
            b.attach(j)
            jobs.append(j)
            bufs.append(b)
        with vf.Batch() as bt:
            assert all(r["status"] == 0 for r in bt.run(jobs))
        return [b.mesh() for b in bufs]

    together = run(range(5))
    for i in range(5):
        alone = run([i])[0]
        np.testing.assert_array_equal(together[i]["xyz"], alone["xyz"])
        np.testing.assert_array_equal(together[i]["tri"], alone["tri"])
