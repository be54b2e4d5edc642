"""cpsd_dev_get into host arrays of the caller's choosing."""
import ctypes as C
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
