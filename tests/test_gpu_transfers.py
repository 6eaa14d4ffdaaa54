"""Transfers of host arrays next to each other (csrc/hostio.h): lattices of one
device share pinned slots."""
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
