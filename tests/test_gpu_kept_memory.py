"""Device memory that a lattice holds between calls (plbamd_set_kept_bytes): bounded,
given back when asked and when an allocation of the library runs short, and
without an effect on the results."""
import contextlib
import ctypes
import threading
import time

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
    """The HIP runtime that the library runs on: torch brings one of its own, which is another if it came later."""
    with open("/proc/self/maps") as maps:
        paths = {line.split()[-1] for line in maps if "libamdhip64" in line}
    path = next((p for p in sorted(paths) if "/torch/" not in p), min(paths))
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


@contextlib.contextmanager
def filled(leave):
    """The device's memory taken but for about `leave` bytes: all that is reported free but 2 GB, then pieces of
    64 MB until there is none (the device has more than it reports), of which `leave` are given back."""
    rt, taken = hip(), []

    def take(n):
        p = ctypes.c_void_p()
        if rt.hipMalloc(ctypes.byref(p), ctypes.c_size_t(n)) != 0:
            return False
        taken.append(p)
        return True
    try:
        assert take(free_bytes() - (2 << 30))
        while take(64 << 20):
            assert len(taken) < 200
        for _ in range(leave // (64 << 20)):
            assert rt.hipFree(taken.pop()) == 0
        yield
    finally:
        rt.hipGetLastError()
        for p in taken:
            assert rt.hipFree(p) == 0


def test_every_allocation_takes_kept_memory_back(gpu, monkeypatch):
    """160^3 FP64: 623 MB of populations and as much kept. With 400 MB left, a probe of 700 MB needs it."""
    monkeypatch.delenv("PLBAMD_FUSED", raising=False)
    with lattice(160) as lat:
        lat.collideAndStream(5)
        assert lat.runInfo()["kept_bytes"] > 590 << 20
        with filled(400 << 20):
            ms, moved, gbs = plb.native.bandwidth_probe("slots", 1400 << 20, repeats=1)
        assert lat.runInfo()["kept_bytes"] == 0


def test_an_allocation_waits_for_the_call_that_uses_kept_memory(gpu, monkeypatch):
    """The same while another thread is in a call of many steps with it: the allocation waits for that call's
    launches instead of failing."""
    monkeypatch.delenv("PLBAMD_FUSED", raising=False)
    with lattice(160) as lat:
        lat.collideAndStream(5)
        with filled(400 << 20):
            t = threading.Thread(target=lat.collideAndStream, args=(12000,))
            t.start()
            time.sleep(0.003)
            with lattice(150) as other:      # 513 MB
                other.collideAndStream(2)
            t.join()
        assert lat.time == 12005
