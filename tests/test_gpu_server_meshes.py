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
