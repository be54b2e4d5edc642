"""Several orbitals per workgroup of the z passes, the V psi pass and the density
pass, with a last group that is not full: every orbital and the density against
the same steps with one orbital per launch.

A z-pass workgroup takes 2 (4) orbitals from 19 (37) at 128^3 and from 33 (65)
at 96^3, a V psi workgroup at 128^3 one for every 8 orbitals, up to 4."""
import numpy as np
import pytest

import cpsd_amd

pytestmark = pytest.mark.gpu


def step(cell, ne, mode, psi, batch, monkeypatch):
    if batch:
        monkeypatch.setenv("CPSD_FFT_BATCH", str(batch))
    else:
        monkeypatch.delenv("CPSD_FFT_BATCH", raising=False)
    dev = cpsd_amd.DeviceSD(cell, ne)
    if mode:
        dev.set_precision(mode)
    dev.set_orbitals(psi)
    dev.run(2, dt=0.5)      # the first step in the mode's precision, the last in FP64
    out = dev.get(c1=True, c2=True, dn=True)
    dev.close()
    return out


@pytest.mark.parametrize("n,ne", [(128, 21), (128, 26), (128, 39), (96, 37), (96, 75)])
def test_groups_of_orbitals(gpu, monkeypatch, n, ne):
    cell = cpsd_amd.water_cell(1, 11.0, n, seed=n)
    psi = cell.random_orbitals(ne, seed=5, decay=0.05)
    # FP64: the two sides add the density in another order, ne 2^-53 of it.  FP32
    # passes: both sides round 24 bits over some 20 operations per axis, against
    # the largest value
    for mode, tol in ((0, 1e-12), (1, 1e-5)):
        print("[gpu-groups] %d^3, %d orbitals, mode %d" % (n, ne, mode), flush=True)
        a = step(cell, ne, mode, psi, 0, monkeypatch)
        b = step(cell, ne, mode, psi, 1, monkeypatch)
        for k in ("c1", "c2"):
            x, y = a[k].reshape(ne, -1), b[k].reshape(ne, -1)
            for i in range(ne):
                assert np.max(np.abs(x[i] - y[i])) < tol * np.max(np.abs(y[i])), (k, i)
        assert np.max(np.abs(a["dn"] - b["dn"])) < tol * np.max(np.abs(b["dn"]))
