"""Meshes of server jobs against a budget that they just fit, beside finished jobs whose grids are still on their way to the
clients."""
import time

import numpy as np
import pytest

from test_gpu_host_copies import Pinned

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
MESH = (96, 96, 96)


def status(vf, budget, job):
    s = vf.Server(budget, 4)
    r = s.wait(s.submit(job))
    s.close()
    return r["status"]


def least_budget(vf, make):
    """The smallest budget (to 64 KiB) with which the job succeeds."""
    lo, hi = 0, 8 << 30
    assert status(vf, hi, make()) == 0
    while hi - lo > 1 << 16:
        mid = (lo + hi) // 2
        if status(vf, mid, make()) == 0:
            hi = mid
        else:
            lo = mid
    return hi


def test_meshes_fit_once_the_grids_before_them_have_left(vf):
    xyz, tri = vf.vessel_mesh(4, *vf.vessel_segments(20000))
    dev = vf.DeviceMesh(xyz, tri)
    dims = (512, 512, 512)  # 268 MB on their way for 5 ms, longer than the other job takes to its meshes
    grid = Pinned(vf, dims)
    buf = vf.MeshBuffers(400000, 800000)

    def large():
        j = dev.job(dims, *BOX, 4, 1, vf.NAIVE, vf.CHEBYSHEV)
        j.labels_out = grid.cells.ctypes.data
        return j

    def meshes():
        j = dev.job(MESH, *BOX, 6, 2, vf.NAIVE, vf.EUCLIDEAN, marching_cubes=1)
        buf.attach(j)
        return j

    alone = least_budget(vf, meshes)
    want = {k: v.copy() for k, v in buf.mesh().items()}
    held = least_budget(vf, large)
    plain = least_budget(vf, lambda: dev.job(MESH, *BOX, 6, 2, vf.NAIVE, vf.EUCLIDEAN))
    budget = max(alone, held + plain) + (1 << 16)
    assert budget < held + alone  # the meshes do not fit beside the large job
    print("budgets", alone, held, plain, budget, flush=True)
    first = None
    for _ in range(3):
        grid.cells[:] = 0
        buf.xyz[:] = 0
        s = vf.Server(budget, 4)
        a = s.submit(large())
        t0 = time.time()
        while s.stats()["in_flight"] == 0 and time.time() - t0 < 5:
            pass
        b = s.submit(meshes())  # admitted when the large job has finished but for its copy
        rb, ra = s.wait(b), s.wait(a)
        s.close()
        assert (ra["status"], rb["status"]) == (0, 0)
        for k, v in buf.mesh().items():
            np.testing.assert_array_equal(v, want[k])
        counts = np.bincount((grid.cells & 0x7FFF).ravel(), minlength=8)
        assert int(counts[2:].sum()) == ra["occupied"]
        first = counts if first is None else first
        np.testing.assert_array_equal(counts, first)
    grid.free()
    dev.close()


def test_smoothing_stays_within_the_reservation(vf):
    # a box of many fragments: nearly all of the job's memory is its meshes' and their smoothing's
    corner = np.array([[x, y, z] for x in (-0.95, 0.95) for y in (-0.95, 0.95) for z in (-0.95, 0.95)], np.float32)
    face = np.array([[0, 1, 3], [0, 3, 2], [4, 6, 7], [4, 7, 5], [0, 4, 5], [0, 5, 1], [2, 3, 7], [2, 7, 6], [0, 2, 6], [0, 6, 4],
                     [1, 5, 7], [1, 7, 3]], np.uint32)
    dev = vf.DeviceMesh(corner, face)
    dims = (100, 96, 104)
    buf = vf.MeshBuffers(1500000, 3000000)

    def job(smooth):
        j = dev.job(dims, *BOX, 250, 3, vf.NAIVE, vf.EUCLIDEAN, marching_cubes=1, smooth=(3, 0.8, 2, 0.3) if smooth else (0, 0, 0, 0))
        buf.attach(j)
        return j

    with vf.Batch() as b:
        assert b.run([job(True)])[0]["status"] == 0
    want = {k: v.copy() for k, v in buf.mesh().items()}
    assert len(want["xyz"]) > 300000
    tight = least_budget(vf, lambda: job(True)) + (1 << 16)
    print("vertices", len(want["xyz"]), "budgets", tight, least_budget(vf, lambda: job(False)), flush=True)
    for budget in (tight, 8 << 30):
        s = vf.Server(budget, 3)
        for _ in range(2):
            buf.xyz[:] = 0
            for smooth in (False, True):
                assert s.wait(s.submit(job(smooth)))["status"] == 0
            for k, v in buf.mesh().items():
                np.testing.assert_array_equal(v, want[k])
        m = s.memory()
        s.close()
        assert m["max_unreserved_bytes"] == 0 and m["reserved_bytes"] == 0 and m["peak_device_bytes"] <= budget, (budget, m)
    dev.close()
