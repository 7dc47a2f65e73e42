"""Results on their way to the caller's memory: grids around the sizes where the copy changes its way, odd addresses and
lengths, several threads at once, pinned memory, and the counts of batch and server jobs with few and many labels."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = ([-1.03, -1.03, -1.03], [1.03, 1.03, 1.03])
# 2 bytes a cell: 1 MiB is where staging starts, 512 KiB a chunk, 2 MiB a launch, 8 MiB the ring of slots
DIMS = [(1, 1, 1), (64, 64, 127), (64, 64, 128), (64, 64, 129), (73, 79, 131), (128, 128, 128), (128, 128, 129),
        (160, 164, 160), (161, 163, 167), (256, 256, 200)]


def cells(dims, seed):
    return np.random.default_rng(seed).integers(0, 0x7FFF, dims, np.uint16)


def read_into(vf, grid, buf):
    vf.check(vf.lib().vf_grid_read(grid._h, C.c_void_p(buf.ctypes.data)))


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("shift", [0, 2, 10])
def test_grid_read(vf, dims, shift):
    print("read", dims, shift, flush=True)
    want = cells(dims, shift)
    n = want.size
    with vf.Grid(dims, *BOX) as g:
        g.write(want)
        room = np.full(n + 64, 0xABCD, np.uint16)
        out = room[shift // 2:shift // 2 + n]
        for _ in range(2):
            read_into(vf, g, out)
            np.testing.assert_array_equal(out, want.ravel())
            assert (room[:shift // 2] == 0xABCD).all() and (room[shift // 2 + n:] == 0xABCD).all()
            out[:] = 0
        np.testing.assert_array_equal(g.occupancy(), (want > 0).astype(np.uint8))


def test_threads_share_the_slots(vf):
    dims = (128, 128, 150)
    grids = [vf.Grid(dims, *BOX) for _ in range(4)]
    want = [cells(dims, 50 + i) for i in range(4)]
    for g, w in zip(grids, want):
        g.write(w)
    bad = []

    def work(i):
        out = np.zeros(dims, np.uint16)
        for _ in range(6):
            out[:] = 0
            read_into(vf, grids[i], out)
            if not (out == want[i]).all():
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in grids:
        g.close()
    assert not bad


class Pinned:
    def __init__(self, vf, dims):
        n = int(np.prod(dims))
        self.lib, self.p = vf.lib(), C.c_void_p()
        assert self.lib.hipHostMalloc(C.byref(self.p), C.c_size_t(2 * n), C.c_uint(0)) == 0
        self.cells = np.ctypeslib.as_array((C.c_uint16 * n).from_address(self.p.value)).reshape(dims)

    def free(self):
        del self.cells
        assert self.lib.hipHostFree(self.p) == 0


def jobs_of(vf, pinned):
    keep, jobs, outs = [], [], []
    xyz, tri = vf.vessel_mesh(3, *vf.vessel_segments(6000))
    dev = vf.DeviceMesh(xyz, tri)
    keep.append(dev)
    for i, (e, seeds, algo) in enumerate([(40, 3, vf.NAIVE), (100, 1500, vf.NAIVE), (96, 20, vf.FLOOD), (33, 1, vf.FLOOD),
                                          (120, 1021, vf.NAIVE), (64, 1022, vf.NAIVE), (64, 1023, vf.NAIVE)]):
        j = dev.job((e, e, e), *BOX, seeds, 7 + i, algo, (vf.EUCLIDEAN, vf.MANHATTAN, vf.CHEBYSHEV)[i % 3])
        if pinned:
            keep.append(Pinned(vf, (e, e, e)))
        lab = keep[-1].cells if pinned else np.empty((e, e, e), np.uint16)
        lab[:] = 0
        hist = np.full(65536, 77, np.uint32)
        j.labels_out, j.histogram_out = lab.ctypes.data, hist.ctypes.data
        outs.append((lab, hist))
        jobs.append(j)
    return jobs, outs, keep


def free(jobs, outs, keep):
    outs.clear()
    for k in keep:
        if isinstance(k, Pinned):
            k.free()


def check(results, outs):
    for r, (lab, hist) in zip(results, outs):
        assert r["status"] == 0
        v = lab & 0x7FFF
        want = np.bincount(v[v > 1], minlength=65536).astype(np.uint32)
        np.testing.assert_array_equal(hist, want)
        assert r["num_labels"] == (want > 0).sum() and int(want.sum()) == r["occupied"]


@pytest.mark.parametrize("pinned", [False, True])
def test_batch_counts_and_grids(vf, pinned):
    jobs, outs, keep = jobs_of(vf, pinned)
    with vf.Batch() as b:
        for _ in range(2):
            check(b.run(jobs), outs)
            for lab, hist in outs:
                lab[:] = 0
                hist[:] = 5
            lab = None
    free(jobs, outs, keep)


@pytest.mark.parametrize("pinned", [False, True])
def test_server_counts_and_grids(vf, pinned):
    print("server", pinned, flush=True)
    jobs, outs, keep = jobs_of(vf, pinned)
    want, wanted, keep2 = jobs_of(vf, False)
    with vf.Batch() as b:
        b.run(want)
    for slots in (64, 2):
        s = vf.Server(64 << 30, slots)
        for _ in range(2):
            tickets = [s.submit(j) for j in jobs]
            check([s.wait(t) for t in tickets], outs)
            for (lab, hist), (ref, _) in zip(outs, wanted):
                np.testing.assert_array_equal(lab, ref)
                lab[:] = 0
                hist[:] = 9
            lab = None
        s.close()
    free(jobs, outs, keep)
