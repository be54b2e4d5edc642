"""The one-workgroup Lagrange fixed point at the edges of its 16 x 16 tiles (1
to 48 orbitals) and the first count above it, over calls that carry the
orbitals on, against the oracle."""
import numpy as np
import pytest

import cpsd_amd
import oracle_lib as O
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ne", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49])
def test_lagrange_by_orbital_count_vs_oracle(gpu, ne):
    print("[gpu-lagrange] %d orbitals at 16^3" % ne, flush=True)
    cell = cpsd_amd.water_cell(1, 11.0, 16, seed=ne)
    psi = cell.random_orbitals(ne, seed=3, decay=0.05)
    st = O.State(O.Setup(1, 11.0, 16, cell.katm, cell.zv), ne, cell.lmmax, cell.vl, cell.vnl, cell.vnlnrm, cell.r, psi,
                 cell.amass)
    dev = cpsd_amd.DeviceSD(cell, ne)
    dev.set_orbitals(psi)
    for _ in range(2):
        Eg, _, _ = dev.run(2)
        Er, _, _ = st.step(2)
        compare(Eg, Er, tol=1e-9)
    o = dev.get(c2=True, lmd=True, hml=True)
    dev.close()
    assert np.max(np.abs(o["c2"] - st.c2)) < 1e-10
    assert np.max(np.abs(o["lmd"] - st.lmd)) < 1e-9
    assert np.max(np.abs(o["hml"] - st.hml)) < 1e-9
