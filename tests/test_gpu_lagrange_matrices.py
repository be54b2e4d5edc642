"""The s matrices that cpsd_dev_debug_fetch 6-9 hands out are those of the last
step, whichever kernel formed them: against the same expressions on the Gram
matrix it hands out as 5 (ccpsdv3/cpsd.c:415-437)."""
import math

import numpy as np
import pytest

import cpsd_amd

pytestmark = pytest.mark.gpu

DT, FMASS = 5.8, 400000.0


def s_matrices(gram, ne, c1_second, dte):
    """s11, s12, s21, s22 with element (r, c) at r + c ne"""
    g = gram.reshape(2 * ne, 2 * ne)
    o1, o2 = (ne, 0) if c1_second else (0, ne)

    def mirrored(rows, cols):    # the upper triangle of a block, mirrored
        u = np.triu(g[rows:rows + ne, cols:cols + ne])
        return u + np.triu(u, 1).T
    g11, g22, g21, g12 = mirrored(o1, o1), mirrored(o2, o2), mirrored(o2, o1), mirrored(o1, o2)
    one = np.eye(ne)
    s21 = (one - g21) * 0.5
    s12 = np.where(one == 1, s21, (one - g12) * 0.5)
    return -g11 * 0.5 * dte, s12, s21, (one - g22) * 0.5 / dte


# 48 is the largest count whose matrices the Lagrange kernel forms itself
@pytest.mark.parametrize("ne", [1, 4, 16, 17, 33, 48, 49])
def test_fetched_s_matrices_are_the_last_steps(gpu, ne):
    print("[gpu-smat] %d orbitals at 24^3" % ne, flush=True)
    cell = cpsd_amd.water_cell(1, 11.0, 24, seed=ne)
    dev = cpsd_amd.DeviceSD(cell, ne)
    # a preconditioned step first, whose matrices are others
    dev.set_preconditioner(np.linspace(0.5, 1.5, cell.nfft3d))
    dev.set_orbitals(cell.random_orbitals(ne, seed=3, decay=0.05))
    dev.run(1, DT, FMASS)
    dev.set_preconditioner(None)
    dev.set_orbitals(cell.random_orbitals(ne, seed=4, decay=0.05))
    for step in range(2):
        dev.run(1, DT, FMASS)
        want = s_matrices(dev.fetch(5), ne, step == 1, DT / math.sqrt(FMASS))
        for what, name, w in zip((6, 7, 8, 9), ("s11", "s12", "s21", "s22"), want):
            if name == "s11" and step == 1:
                continue     # <c1|c1> is carried from the first step, not formed again
            got = dev.fetch(what)
            # the same operations on the same numbers: a few roundings at most
            assert np.max(np.abs(got - w.ravel(order="F"))) <= 4 * np.finfo(float).eps * np.max(np.abs(w)), (name, step)
    dev.close()
