"""Host copies through the pinned ring: arrays just below and above its
smallest size, with a last chunk that is not whole, and larger than the ring,
come back as they went up, from several threads at once too."""
import threading

import numpy as np
import pytest

import cpsd_amd

pytestmark = pytest.mark.gpu


def round_trip(ne, seed):
    cell = cpsd_amd.water_cell(1, 14.0, 48, seed=1)
    psi = cell.random_orbitals(ne, seed=seed, decay=0.05)
    dev = cpsd_amd.DeviceSD(cell, ne)
    for k in (1.0, 2.0):          # the second use of the ring
        dev.set_orbitals(k * psi)
        assert np.array_equal(dev.get(c2=True)["c2"].ravel(), (k * psi).ravel())
    dev.close()


# 0.92 MB per orbital; the ring takes arrays from 4 MB, in chunks of 2, 16 in all
@pytest.mark.parametrize("ne", [4, 5, 18, 41])
def test_round_trip_by_size(gpu, ne):
    print("[gpu-copies] %d orbitals at 48^3" % ne, flush=True)
    round_trip(ne, 3)


def test_round_trip_threads(gpu):
    print("[gpu-copies] three contexts, three threads", flush=True)
    bad = []

    def one(seed):
        try:
            round_trip(20, seed)
        except BaseException as e:   # noqa: BLE001
            bad.append(e)
    th = [threading.Thread(target=one, args=(s,)) for s in (5, 6, 7)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
