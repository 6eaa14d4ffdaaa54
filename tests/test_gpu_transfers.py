"""Transfers of host arrays next to each other (csrc/hostio.h): lattices of one
device share pinned slots."""
import threading

import numpy as np
import pytest

import palabos_amd as plb
from cases import uniform

pytestmark = pytest.mark.gpu


def lattice(shape):
    return plb.Block3D(*shape, plb.D3Q19, plb.BGK(1.7), storage="f64", periodic=True)


def test_without_pinned_memory_beside_a_lattice_that_has_it(gpu, monkeypatch):
    """PLBAMD_NO_PINNED counts at every transfer, also when another lattice, or this one, holds the device's slots."""
    shape = (9, 8, 7)
    f = 0.02 * uniform(shape + (19,), 3)
    with lattice(shape) as other, lattice(shape) as lat:
        for q in (other, lat):
            q.setPopulations(f)
            assert q.runInfo()["pinned_transfers"] == 1 and q.runInfo()["pageable_transfers"] == 0
        monkeypatch.setenv("PLBAMD_NO_PINNED", "1")
        with lattice(shape) as third:
            for q in (lat, third):
                q.setPopulations(2 * f)
                assert np.array_equal(q.getPopulations(), 2 * f)
                assert q.runInfo()["pageable_transfers"] == 2
            assert third.runInfo()["pinned_transfers"] == 0
        monkeypatch.delenv("PLBAMD_NO_PINNED")
        assert np.array_equal(lat.getPopulations(), 2 * f)
        assert lat.runInfo()["pinned_transfers"] == 2


def test_a_small_read_does_not_wait_for_another_lattices_transfer(gpu):
    """One cell's read waits for a chunk of the other transfer (4 MB), not for its 1.3 GB of populations."""
    with lattice((204, 204, 204)) as big, lattice((8, 8, 8)) as small:
        small.macroscopic((1, 1, 1, 1, 1, 1))
        big.getPopulations((0, 0, 0, 203, 0, 203))
        done = threading.Event()

        def transfer():
            try:
                big.getPopulations()
            finally:
                done.set()
        t = threading.Thread(target=transfer)
        reads = 0
        t.start()
        while not done.is_set():
            small.macroscopic((1, 1, 1, 1, 1, 1))
            reads += 1
        t.join()
        print(f"[transfers] {reads} reads beside one transfer", flush=True)
        assert reads >= 10   # some hundred; one or two when they wait for all of it


def test_transfers_of_many_threads(gpu):
    """More transfers at once than there are slots, each of several chunks: every array arrives whole."""
    shape, n = (40, 64, 96), 12
    lats = [lattice(shape) for _ in range(n)]
    try:
        f = [0.02 * uniform(shape + (19,), 5 + k) for k in range(n)]
        wrong = []

        def go(k):
            for _ in range(3):
                lats[k].setPopulations(f[k])
                if not np.array_equal(lats[k].getPopulations(), f[k]):
                    wrong.append(k)
        threads = [threading.Thread(target=go, args=(k,)) for k in range(n)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert wrong == []
    finally:
        for lat in lats:
            lat.close()


@pytest.mark.parametrize("shape", [(6, 70, 75), (100, 80, 66), (2, 801, 327), (1, 9, 63000)])
def test_uploads_by_size(gpu, shape):
    """Populations of 4.8 MB (one copy to the device) and of 80 to 86 MB, whose chunks in pinned memory are whole
    x planes, rows of one plane and parts of one row: every value arrives, in a box that starts off the edges too."""
    with lattice(shape) as lat:
        f = 0.02 * uniform(shape + (19,), 3)
        lat.setPopulations(f)
        pinned = f.nbytes >= 72 * 2 ** 20
        assert lat.runInfo()["pinned_transfers"] == int(pinned)
        assert lat.runInfo()["pageable_transfers"] == int(not pinned)
        assert np.array_equal(lat.getPopulations(), f)
        x0, y0, z0 = (n // 3 for n in shape)
        part = 0.02 * uniform(f[x0:, y0:, z0:].shape, 4)
        f[x0:, y0:, z0:] = part
        lat.setPopulations(part, (x0, shape[0] - 1, y0, shape[1] - 1, z0, shape[2] - 1))
        assert np.array_equal(lat.getPopulations(), f)
        lat.initializeAtEquilibrium(1.0 + 0.01 * uniform(shape, 5), 0.02 * uniform(shape + (3,), 6))
        rho, u = lat.macroscopic()
        np.testing.assert_allclose(rho, 1.0 + 0.01 * uniform(shape, 5), rtol=1e-13)
        np.testing.assert_allclose(u, 0.02 * uniform(shape + (3,), 6), rtol=1e-9, atol=1e-14)
