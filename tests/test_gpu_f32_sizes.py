"""The FP32 projection and apply at the edges of their orbital tiles (32, 64,
128) and projector tiles (64, 96, 128), with and without the preconditioned
update, against the FP64 steps."""
import numpy as np
import pytest

import cpsd_amd

pytestmark = pytest.mark.gpu


def kinetic_factors(cell):
    """1 at G = 0 falling with the kinetic energy, one factor per half-complex G"""
    return 1.0 / (1.0 + 0.2 * cell.tg)


# molecules (6 projectors each), orbitals.  FP32 products of 24 bits over some tens to hundreds of terms, two steps
@pytest.mark.parametrize("precond", [0, 1])
@pytest.mark.parametrize("nmol,ne", [(3, 17), (10, 32), (11, 33), (16, 64), (17, 65), (21, 31), (22, 129)])
def test_f32_products_by_size(gpu, nmol, ne, precond):
    print("[gpu-f32] %d projectors, %d orbitals at 16^3, preconditioner %d" % (6 * nmol, ne, precond), flush=True)
    cell = cpsd_amd.water_cell(nmol, 14.0, 16, seed=nmol)
    psi = cell.random_orbitals(ne, seed=3, decay=0.05)
    out = []
    for mode in (0, 1):
        dev = cpsd_amd.DeviceSD(cell, ne)
        dev.set_orbitals(psi)
        if precond:
            dev.set_preconditioner(kinetic_factors(cell))
        dev.run(1)
        dev.set_precision(mode)
        dev.run(3)
        out.append(dev.get(c2=True)["c2"])
        dev.close()
    assert np.max(np.abs(out[0] - out[1])) < 1e-5 * np.max(np.abs(out[0]))
