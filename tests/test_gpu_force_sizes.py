"""Moving ions at the edges of the force kernels: ion counts around the 32 ions
that one pass of the pair sums holds, and projector counts that leave the
column tiles of the nonlocal force partly empty, against the oracle."""
import numpy as np
import pytest

import cpsd_amd
import oracle_lib as O
from test_gpu_forces import say
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


# molecules (3 ions and 6 projectors each), orbitals
@pytest.mark.parametrize("nmol,ne", [(1, 3), (10, 17), (11, 40), (22, 9), (24, 66)])
def test_forces_by_ion_count_vs_oracle(gpu, nmol, ne):
    say("device move=1, %d ions, %d orbitals at 16^3" % (3 * nmol, ne))
    cell = cpsd_amd.water_cell(nmol, 14.0, 16, seed=nmol)
    psi = cell.random_orbitals(ne, seed=3, decay=0.05)
    st = O.State(O.Setup(1, 14.0, 16, cell.katm, cell.zv), ne, cell.lmmax, cell.vl, cell.vnl, cell.vnlnrm, cell.r,
                 psi, cell.amass)
    dev = cpsd_amd.DeviceSD(cell, ne)
    dev.set_ions(1)
    dev.set_orbitals(psi)
    Eg, _, _ = dev.run(2)
    Er, _, _ = st.step(2, move=1)
    compare(Eg, Er)
    ions = dev.get_ions()
    # relative to the largest force: the pairs of a dense random cell are close
    assert np.max(np.abs(ions["fion"] - st.fion)) < 1e-9 * max(1.0, np.max(np.abs(st.fion)))
    assert np.max(np.abs(ions["r2"] - st.r2)) < 1e-12 * max(1.0, np.max(np.abs(st.r2)))
    dev.close()
