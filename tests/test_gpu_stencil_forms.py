"""Erosion and isolated cells on both sides of the lines between the stencils that go by bricks and by cells: thin grids
along each axis, grids of few and of many bricks, one of a batch.  Cells equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from test_gpu_stencils import labelled

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
# bricks of 8 x 8 x 32: 72 and 100 (windows above 3 from 64 on), 300 and 336 (window 3 from 320), 605 and 660 (isolated
# cells from 640), 975 and 1020; then grids whose cells are less than a third of their bricks'
DIMS = [(47, 48, 41), (80, 80, 31), (80, 80, 70), (90, 60, 97), (88, 83, 130), (88, 90, 130), (100, 115, 130), (136, 117, 97), (61, 65, 3), (1, 130, 200), (150, 2, 90),
        (300, 70, 10), (300, 70, 11)]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("kind,size", [(2, 3), (0, 5), (1, 7)])
def test_windows(vf, dims, kind, size):
    print("erode", dims, kind, size, flush=True)
    grid = labelled(dims, sum(dims) + size)
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        g.erode(kind, size, 2, 0.6, 0.8, 77)
        want = O.erode(grid.copy(), kind, size, 2, 0.6, 0.8, 77)
        np.testing.assert_array_equal(g.read(), want)
        assert g.count_occupied() == int((want != 0).sum())


@pytest.mark.parametrize("dims", DIMS)
def test_isolated_cells(vf, dims):
    grid = labelled(dims, sum(dims))
    with vf.Grid(dims, *BOX) as g:
        g.write(grid)
        g.remove_isolated_cells()
        np.testing.assert_array_equal(g.read(), O.remove_isolated_cells(grid))


def test_a_batch_with_both(vf):
    xyz, tri = vf.vessel_mesh(9, *vf.vessel_segments(8000))
    mesh = vf.DeviceMesh(xyz, tri)
    jobs, outs = [], []
    for dims in ((40, 40, 40), (100, 100, 100), (120, 110, 6)):
        j = mesh.job(dims, *BOX, 7, 3, vf.NAIVE, vf.EUCLIDEAN)
        j.erode, j.erosion_convolution, j.erosion_size, j.erosion_iterations = 1, vf.EROSION_ELLIPSE, 3, 2
        j.erosion_probability, j.erosion_threshold, j.erosion_seed = 0.5, 0.5, 11
        out = np.zeros(dims, np.uint16)
        j.labels_out = out.ctypes.data
        jobs.append(j)
        outs.append(out)
    with vf.Batch() as b:
        results = b.run(jobs)
    for r, j, out in zip(results, jobs, outs):
        dims = out.shape
        assert r["status"] == 0
        occ = O.voxelize(xyz, tri, *BOX, dims)
        want = O.erode(O.naive(occ, O.seed_uniform(occ, 7, 3), vf.EUCLIDEAN), vf.EROSION_ELLIPSE, 3, 2, 0.5, 0.5, 11)
        np.testing.assert_array_equal(out, want)
    mesh.close()


def test_a_flat_grid_takes_no_bricks(vf):
    import time
    dims = (2048, 2048, 1)
    grid = (np.random.default_rng(0).random(dims) < 0.2).astype(np.uint16)
    took = []
    with vf.Grid(dims, *BOX) as g:
        for _ in range(6):
            g.write(grid)
            t0 = time.perf_counter()
            g.remove_isolated_cells()
            took.append(time.perf_counter() - t0)
        np.testing.assert_array_equal(g.read(), O.remove_isolated_cells(grid))
    print("isolated cells of a flat grid:", min(took), flush=True)
    assert min(took) < 300e-6  # 700 us by bricks, of whose 2048 cells it has 64 each; 95
