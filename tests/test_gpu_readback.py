"""cpsd_dev_get into host arrays of the caller's choosing."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import cpsd_amd

pytestmark = pytest.mark.gpu


def resident(ne, n=48, steps=2):
    """a context of `ne` orbitals (0.92 MB each at 48^3) whose c1, c2 and cpsi differ"""
    cell = cpsd_amd.water_cell(1, 14.0, n, seed=1)
    dev = cpsd_amd.DeviceSD(cell, ne)
    dev.set_orbitals(cell.random_orbitals(ne, seed=3, decay=0.05))
    dev.run(steps)
    return dev


def get(dev, c1=None, c2=None, cpsi=None, dn=None):
    p = [a.ctypes.data_as(C.c_void_p) if a is not None else None for a in (c1, c2, cpsi, dn)]
    assert cpsd_amd.hip_lib().cpsd_dev_get(dev.h, *p, None, None) == 0


# arrays of two and three of the ring's 2 MB chunks: the next array's first chunk
# is on its way while they are still being emptied
@pytest.mark.parametrize("ne", [5, 6])
def test_one_array_passed_twice_holds_the_last(gpu, ne):
    print("[gpu-readback] %d orbitals, c1 and c2 into one array" % ne, flush=True)
    dev = resident(ne)
    size = ne * dev.cell.n2ft3d
    c2, dn = np.empty(size), np.empty(dev.cell.n2ft3d)
    get(dev, c2=c2)
    get(dev, dn=dn)
    for _ in range(300):
        both = np.empty(size)
        get(dev, c1=both, c2=both)
        assert np.array_equal(both, c2)
    for _ in range(100):
        both = np.empty(size)
        get(dev, c1=np.empty(size), c2=both, dn=both)
        assert np.array_equal(both[:dn.size], dn) and np.array_equal(both[dn.size:], c2[dn.size:])
    dev.close()


class Hip:
    """as much of the HIP runtime as the tests need"""

    def __init__(self):
        self.L = C.CDLL("libamdhip64.so")
        for f in ("hipMalloc", "hipHostMalloc", "hipMemcpy", "hipFree", "hipHostFree"):
            getattr(self.L, f).restype = C.c_int

    def ok(self, rc, what):
        assert rc == 0, "%s failed: %d" % (what, rc)

    def device(self, nbytes):
        p = C.c_void_p()
        self.ok(self.L.hipMalloc(C.byref(p), C.c_size_t(nbytes)), "hipMalloc")
        return p

    def pinned(self, size):
        """the address and an array of `size` doubles"""
        p = C.c_void_p()
        self.ok(self.L.hipHostMalloc(C.byref(p), C.c_size_t(8 * size), C.c_uint(0)), "hipHostMalloc")
        return p, np.frombuffer((C.c_double * size).from_address(p.value), dtype=np.float64)

    def download(self, host, dev, nbytes):
        self.ok(self.L.hipMemcpy(host, dev, C.c_size_t(nbytes), 2), "hipMemcpy")


def test_pinned_arrays_take_the_direct_copy(gpu):
    """as fast as the bare copy of the same bytes, give or take the unpacking and
    the call (by the ring it takes 1.5 times as long)"""
    dev = resident(64)
    size = 64 * dev.cell.n2ft3d
    want = np.empty(size)
    get(dev, c2=want)
    hip = Hip()
    ph, host = hip.pinned(size)
    pd = hip.device(8 * size)

    def best(f):
        t = []
        for _ in range(20):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        return min(t)
    tc, tg = best(lambda: hip.download(ph, pd, 8 * size)), best(lambda: get(dev, c2=host))
    print("[gpu-readback] 59 MB to pinned memory: copy %.3f ms, get %.3f ms" % (1e3 * tc, 1e3 * tg), flush=True)
    assert np.array_equal(host, want)
    assert tg < 1.25 * tc
    # one of three arrays pinned, the others through the ring
    a, b = np.empty(size), np.empty(size)
    host[:] = 0.0
    get(dev, c1=a, c2=host, cpsi=b)
    ref = dev.get(c1=True, c2=True, cpsi=True)
    assert np.array_equal(a, ref["c1"]) and np.array_equal(host, ref["c2"]) and np.array_equal(b, ref["cpsi"])
    dev.close()
    hip.ok(hip.L.hipFree(pd), "hipFree")
    hip.ok(hip.L.hipHostFree(ph), "hipHostFree")


def fill(dev, ne, names):
    return {k: np.full(ne * dev.cell.n2ft3d, np.nan) for k in names}


# one array on either side of the 8 MB from which a call is staged (9 and 10
# orbitals are 8.3 and 9.2 MB, the line lies at 8.4), of more than the ring, and
# with a last chunk that is not whole; three arrays of 3.7 MB (a staged call whose
# arrays are each below 4 MB), of 4.6 (each staged) and of 14.7.
@pytest.mark.parametrize("ne,names", [(9, ("c2",)), (10, ("c2",)), (18, ("c2",)), (41, ("c2",)),
                                      (4, ("c1", "c2", "cpsi")), (5, ("c1", "c2", "cpsi")), (16, ("c1", "c2", "cpsi")),
                                      (5, ("c1", "cpsi"))])
def test_read_back_by_size(gpu, ne, names):
    print("[gpu-readback] %d orbitals at 48^3, %s" % (ne, " ".join(names)), flush=True)
    dev = resident(ne)
    dev.run(3)
    blocks = dev.fetch(11).reshape(2, -1)   # the packed G coefficients; after 5 steps c1's are the first
    packed = dict(c1=blocks[0], c2=blocks[1], cpsi=dev.fetch(3))
    mask = dev.cell.masker.reshape(-1, 2)[:, 0] != 0
    ngp = dev.sizes()["ngp"]
    for _ in range(2):
        out = fill(dev, ne, names)
        get(dev, **out)
        for k in names:
            full = out[k].reshape(ne, -1, 2)
            want = packed[k].reshape(ne, ngp, 2)[:, :mask.sum()]
            assert np.array_equal(full[:, mask], want), k
            assert not np.any(full[:, ~mask]), k
    dev.close()


def test_read_back_in_more_threads_than_rings(gpu):
    """six contexts read back at once (four rings at most, one kept between the
    contexts), freed and made again"""
    print("[gpu-readback] six contexts, six threads", flush=True)
    bad = []

    def one(seed):
        try:
            for rep in range(2):
                cell = cpsd_amd.water_cell(1, 14.0, 48, seed=1)
                dev = cpsd_amd.DeviceSD(cell, 20)
                for k in (1.0, 2.0, 3.0, 4.0):
                    psi = k * cell.random_orbitals(20, seed=seed, decay=0.05)
                    dev.set_orbitals(psi)
                    assert np.array_equal(dev.get(c2=True)["c2"], psi.ravel())
                dev.close()
        except BaseException as e:   # noqa: BLE001
            bad.append(e)
    th = [threading.Thread(target=one, args=(s,)) for s in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


def pinned_rings():
    """mappings of this process of a ring's size on the GPU's device file"""
    n = 0
    with open("/proc/self/maps") as f:
        for line in f:
            lo, hi = line.split()[0].split("-")
            n += "/dev/dri/" in line and int(hi, 16) - int(lo, 16) == 8 << 20
    return n


def test_contexts_share_the_ring(gpu):
    """read-backs one after the other leave as many 8 MB pinned as the first,
    whatever the number of contexts, and a context that goes takes none away
    from those that stay"""
    devs = [resident(12) for _ in range(6)]
    want = devs[0].get(c2=True)["c2"]
    first = pinned_rings()
    for d in devs[1:]:
        assert np.array_equal(d.get(c2=True)["c2"], want)
    print("[gpu-readback] 8 MB mappings after the first read-back %d, after six contexts' %d"
          % (first, pinned_rings()), flush=True)
    assert pinned_rings() == first
    for d in devs[:-1]:
        d.close()
    assert np.array_equal(devs[-1].get(c2=True)["c2"], want)
    devs[-1].close()


def test_refused_read_backs_leave_the_next_ones_whole(gpu):
    """while a stream is captured in global mode the runtime refuses the call's
    wait, so it fails, with its copies on their way; more often than there are rings"""
    print("[gpu-readback] refused during a capture", flush=True)
    devs = [resident(20), resident(20, steps=3)]
    want = [d.get(c2=True)["c2"] for d in devs]
    hip = Hip()
    for _ in range(6):
        s, g = C.c_void_p(), C.c_void_p()
        hip.ok(hip.L.hipStreamCreate(C.byref(s)), "hipStreamCreate")
        hip.ok(hip.L.hipStreamBeginCapture(s, 0), "hipStreamBeginCapture")
        a = np.empty_like(want[0])
        p = [None, a.ctypes.data_as(C.c_void_p), None, None, None, None]
        assert cpsd_amd.hip_lib().cpsd_dev_get(devs[0].h, *p) == -1
        hip.L.hipStreamEndCapture(s, C.byref(g))     # invalidated by the call
        hip.L.hipGetLastError()
        hip.ok(hip.L.hipStreamDestroy(s), "hipStreamDestroy")
        for d, w in zip(devs, want):
            assert np.array_equal(d.get(c2=True)["c2"], w)
    for d in devs:
        d.close()
    dev = resident(20)
    assert np.array_equal(dev.get(c2=True)["c2"], want[0])
    dev.close()
