"""Single-grid calls that end in an error, and the grid afterwards."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
EUC, MAN, CHE = 0, 1, 2


def winding_path(dims):
    """One corridor, a cell wide, through the whole grid: along x, row after row, layer after layer."""
    nx, ny, nz = dims
    g = np.zeros(dims, np.uint16)
    g[:, ::2, ::2] = 1
    rows, layers = (ny + 1) // 2, (nz + 1) // 2
    for k in range(layers):
        for r in range(rows - 1):  # the ends of the rows, in turn
            g[-1 if (k * rows + r) % 2 == 0 else 0, 2 * r + 1, 2 * k] = 1
        if k + 1 < layers:  # a layer ends where the next begins
            g[-1 if (k * rows + rows - 1) % 2 == 0 else 0, 2 * (rows - 1) if k % 2 == 0 else 0, 2 * k + 1] = 1
    return g


def overlong_flood(g):
    """A flood whose distances do not fit its keys: 4096 seeds take 12 bits, which leaves a distance 18, and the path of
    about 190000 cells of weight 2 on average is longer than 2^18."""
    seeds = np.zeros((4096, 4), np.uint32)
    seeds[:, 3] = 2 + np.arange(4096) % 250
    g.fracture_flood(seeds, MAN, noise_seed=5, noise_amp=2)


LONG = (96, 88, 88)


def test_flood_after_one_that_failed(vf):
    # rounds are queued ahead: none of the failed flood's may be left when the next one on the grid begins
    path = winding_path(LONG)
    seeds = np.array([[0, 0, 0, 2], [50, 40, 44, 3], [95, 44, 20, 4]], np.uint32)
    want = O.flood(path, seeds, 6, 3, 1)
    with vf.Grid(LONG, *BOX) as g:
        g.write(path)
        for _ in range(3):
            with pytest.raises(vf.VfError, match="VF_ERR_OVERFLOW"):
                overlong_flood(g)
            for _ in range(2):
                g.fracture_flood(seeds, MAN, noise_seed=3, noise_amp=1)
                np.testing.assert_array_equal(g.read(), want)


def test_a_failed_flood_leaves_the_labels(vf):
    path = winding_path(LONG)
    path[10:20, ::2, ::2] = 0x8007  # cells of a fragment, flagged
    path[:, 0, 0] = 5
    seeds = np.array([[0, 0, 0, 2], [50, 40, 44, 3]], np.uint32)
    with vf.Grid(LONG, *BOX) as g:
        g.write(path)
        mesh = g.marching_cubes(7)
        with pytest.raises(vf.VfError, match="VF_ERR_OVERFLOW"):
            overlong_flood(g)
        np.testing.assert_array_equal(g.read(), path)
        np.testing.assert_array_equal(g.occupancy(), (path != 0).astype(np.uint8))
        np.testing.assert_array_equal(g.histogram(), O.histogram(path))
        np.testing.assert_array_equal(g.read_mesh()["xyz"], mesh["xyz"])
        g.homogenize()  # labels of one flood, kept by a failed one after it
        g.fracture_flood(seeds, MAN, noise_seed=3, noise_amp=1)
        want = O.flood((path != 0).astype(np.uint16), seeds, 6, 3, 1)
        with pytest.raises(vf.VfError, match="VF_ERR_OVERFLOW"):
            overlong_flood(g)
        np.testing.assert_array_equal(g.read(), want)


@pytest.mark.parametrize("read_first", [False, True])
def test_a_failed_voxelization_of_a_new_box_leaves_it_empty(vf, read_first):
    dims = (40, 33, 50)
    xyz, tri = vf.vessel_mesh(5, *vf.vessel_segments(3000))
    bad = tri.copy()
    bad[len(tri) // 2, 1] = len(xyz)  # found on the device only
    good, broken = vf.DeviceMesh(xyz, tri), vf.DeviceMesh(xyz, bad)
    empty = np.zeros(dims, np.uint16)
    want = O.voxelize(xyz, tri, *BOX, dims)
    with vf.Grid(dims, *BOX) as g:
        for _ in range(2):
            if read_first:
                np.testing.assert_array_equal(g.read(), empty)
            with pytest.raises(vf.VfError, match="VF_ERR_INVALID_ARG"):
                g.voxelize_device(broken)
            np.testing.assert_array_equal(g.read(), empty)
            np.testing.assert_array_equal(g.histogram(), np.zeros(65536, np.uint32))
            g.voxelize_device(good)
            np.testing.assert_array_equal(g.read(), want)
            with pytest.raises(vf.VfError, match="VF_ERR_INVALID_ARG"):  # a grid with values keeps them
                g.voxelize_device(broken)
            np.testing.assert_array_equal(g.read(), want)
            np.testing.assert_array_equal(g.occupancy(), want)
            g.set_aabb(*BOX, dims)
    good.close()
    broken.close()
