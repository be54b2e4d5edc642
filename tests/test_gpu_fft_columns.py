"""The transforms' packed columns: every grid's cutoff disc (row lengths that
are no multiple of a line, column counts that leave the last z workgroup partly
empty), a mask whose rows reach the Nyquist column, orbital counts around the
orbitals one workgroup takes, and the FP32 passes, against the oracle and the
FP64 passes."""
import numpy as np
import pytest

import cpsd_amd
import oracle_lib as O
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


def nyquist_rows(cell, setup):
    """fill the rows ky = kz = 0 and ky = 1, kz = N - 2 up to kx = N/2"""
    n = cell.nfft
    for masker in (cell.masker, setup.masker):
        m = masker.reshape(n, n, n // 2 + 1, 2)
        m[0, 0] = 1
        m[n - 2, 1] = 1


def cell_and_oracle(n, ne, nyq):
    cell = cpsd_amd.water_cell(1, 11.0, n, seed=n)
    setup = O.Setup(1, 11.0, n, cell.katm, cell.zv)
    if nyq:
        nyquist_rows(cell, setup)
    psi = cell.random_orbitals(ne, seed=5, decay=0.05)
    st = O.State(setup, ne, cell.lmmax, cell.vl, cell.vnl, cell.vnlnrm, cell.r, psi, cell.amass)
    return cell, psi, st


@pytest.mark.parametrize("n,ne,nyq", [(8, 3, 0), (12, 5, 0), (16, 4, 0), (16, 4, 1), (20, 3, 0), (24, 3, 1), (32, 7, 0), (40, 3, 0),
                                      (48, 2, 1), (64, 2, 0), (80, 2, 0), (96, 2, 1), (128, 1, 0), (128, 5, 1)])
def test_step_by_grid_vs_oracle(gpu, n, ne, nyq):
    print("[gpu-columns] %d^3, %d orbitals, Nyquist rows %d" % (n, ne, nyq), flush=True)
    cell, psi, st = cell_and_oracle(n, ne, nyq)
    dev = cpsd_amd.DeviceSD(cell, ne)
    dev.set_orbitals(psi)
    Eg, _, _ = dev.run(2)
    Er, _, _ = st.step(2)
    compare(Eg, Er, tol=1e-9)
    o = dev.get(c2=True, dn=True)
    dev.close()
    assert np.max(np.abs(o["dn"] - st.dn)) < 1e-10
    assert np.max(np.abs(o["c2"] - st.c2)) < 1e-10


# FP32 transforms: 24 bits over some 20 dependent roundings per axis, against the largest value
@pytest.mark.parametrize("n,ne", [(8, 3), (20, 4), (48, 5), (64, 3), (80, 9), (96, 2), (128, 6)])
def test_fp32_passes_vs_fp64(gpu, n, ne):
    print("[gpu-columns] FP32 %d^3, %d orbitals" % (n, ne), flush=True)
    cell = cpsd_amd.water_cell(1, 11.0, n, seed=n)
    psi = cell.random_orbitals(ne, seed=5, decay=0.05)
    out = []
    for mode in (0, 1):
        dev = cpsd_amd.DeviceSD(cell, ne)
        dev.set_precision(mode)
        dev.set_orbitals(psi)
        dev.run(2)
        out.append(dev.get(c2=True, dn=True))
        dev.close()
    for k in ("c2", "dn"):
        assert np.max(np.abs(out[0][k] - out[1][k])) < 1e-5 * np.max(np.abs(out[0][k])), k
