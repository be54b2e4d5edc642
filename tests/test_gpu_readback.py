"""cpsd_dev_get into host arrays of the caller's choosing."""
import ctypes as C

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
