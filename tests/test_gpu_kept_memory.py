"""Device memory that a lattice holds between calls (plbamd_set_kept_bytes): bounded,
given back when asked and when an allocation of the library runs short, and
without an effect on the results."""
import ctypes

import numpy as np
import pytest

import palabos_amd as plb
from cases import uniform

pytestmark = pytest.mark.gpu


def lattice(n, storage="f64", periodic=True):
    lat = plb.Block3D(n, n, n, plb.D3Q19, plb.BGK(1.7), storage=storage, periodic=periodic)
    lat.toggleInternalStatistics(False)
    return lat


def hip():
    """The HIP runtime that the library runs on."""
    with open("/proc/self/maps") as maps:
        path = next(line.split()[-1] for line in maps if "libamdhip64" in line)
    return ctypes.CDLL(path)


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_kept_bytes_are_bounded_and_given_back(gpu, monkeypatch):
    monkeypatch.delenv("PLBAMD_FUSED", raising=False)
    n = 128
    array = 19 * 8 * n ** 3
    with lattice(n, periodic=False) as lat:
        u = 0.02 * uniform((n, n, n, 3), 3)
        lat.initializeAtEquilibrium(1.0, u)
        assert lat.runInfo()["kept_bytes"] == 0
        lat.collideAndStream(5)
        info = lat.runInfo()
        assert info["two_step_launches"] == 2 and array <= info["kept_bytes"] <= array + 8 * n ** 3 + (1 << 20)
        before = free_bytes()
        lat.setKeptBytes(0)
        assert lat.runInfo()["kept_bytes"] == 0
        assert free_bytes() - before >= array
        lat.collideAndStream(4)                      # one step per launch
        assert lat.runInfo()["two_step_launches"] == 2 and lat.runInfo()["kept_bytes"] == 0
        lat.setKeptBytes(array)                      # without room for the words of the edges
        lat.collideAndStream(4)
        assert lat.runInfo()["two_step_launches"] == 2
        lat.setKeptBytes(-1)
        lat.collideAndStream(4)
        assert lat.runInfo()["two_step_launches"] == 4 and lat.runInfo()["kept_bytes"] == info["kept_bytes"]
        got = lat.getPopulations()
    monkeypatch.setenv("PLBAMD_FUSED", "0")
    with lattice(n, periodic=False) as lat:
        lat.initializeAtEquilibrium(1.0, u)
        lat.collideAndStream(17)
        assert np.array_equal(lat.getPopulations(), got)


def test_adjoint_buffer_keeps_to_the_budgets(gpu):
    n = 24

    def gradient(lat):
        lat.setPorosity(0.3 * uniform((n, n, n), 5) ** 2)
        lat.initializeAtEquilibrium(1.0, (0.01, 0.0, 0.0))
        return lat.adjointGradient(20, 10, 1, n - 2)[1]
    with lattice(n) as lat:
        want = gradient(lat)
        held = lat.runInfo()["kept_bytes"]
        assert held > 0
        lat.setAdjointRecordBytes(0)                 # a budget of the caller: nothing larger is kept
        assert np.array_equal(gradient(lat), want)
        assert lat.runInfo()["kept_bytes"] == 0
        lat.setAdjointRecordBytes(held)
        assert np.array_equal(gradient(lat), want)
        assert 0 < lat.runInfo()["kept_bytes"] <= held
        lat.setKeptBytes(held // 4)
        assert lat.runInfo()["kept_bytes"] == 0
        assert np.array_equal(gradient(lat), want)
        assert lat.runInfo()["kept_bytes"] == 0
        lat.setKeptBytes(-1)
        lat.setAdjointRecordBytes(-1)
        assert np.array_equal(gradient(lat), want)
        assert lat.runInfo()["kept_bytes"] == held
    with pytest.raises(plb.native.PlbError):
        lattice(8).setKeptBytes(-2)
