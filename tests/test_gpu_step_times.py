"""Times of steps against each other, where a slip of the compiler or of the set-up
has cost a fifth and more before. Best of several runs in one process, with room
for the noise of small ratios."""
import pytest

import palabos_amd as plb

pytestmark = pytest.mark.gpu


def step_us(lat, steps, repeats=6):
    lat.toggleInternalStatistics(False)
    lat.collideAndStream(9)
    return min(lat.collideAndStreamTimed(steps) for _ in range(repeats)) * 1e3 / steps


def test_tagged_odd_steps_keep_their_loads_together(gpu, monkeypatch):
    """Odd nz in 16-bit storage takes the unstaged kernel. With tags it reads one byte a
    cell more than without (1/38 of its traffic) and tests it: 1.11 times the time, and
    1.24 times with a wait after each of the loads."""
    monkeypatch.setenv("PLBAMD_FUSED", "0")
    monkeypatch.setenv("PLBAMD_CACHED_Z", "1")
    shape, us = (191, 203, 197), []
    for tagged in (False, True):
        with plb.Block3D(*shape, plb.D3Q19, plb.BGK(1.8), storage="bf16", periodic=True) as lat:
            if tagged:
                lat.defineDynamics((0, 0, 0, shape[1] - 1, 0, shape[2] - 1), plb.BounceBack)
            us.append(step_us(lat, 50))
    print(f"[step time] plain {us[0]:.1f} us, tagged {us[1]:.1f} us", flush=True)
    assert us[1] < 1.17 * us[0]


def test_timed_steps_do_not_include_their_set_up(gpu, monkeypatch):
    """The first timed call of a lattice allocates the second array and its tables (a millisecond and more) before the
    clock starts, as any later one finds them."""
    monkeypatch.delenv("PLBAMD_FUSED", raising=False)

    def first_and_next():
        with plb.Block3D(128, 128, 128, plb.D3Q19, plb.BGK(1.8), storage="f64") as lat:
            lat.toggleInternalStatistics(False)
            lat.collideAndStream(1)
            first = lat.collideAndStreamTimed(4)
            assert lat.runInfo()["two_step_launches"] == 2
            return first, min(lat.collideAndStreamTimed(4) for _ in range(5))
    first_and_next()     # the kernels' code comes with the first use in a process
    first, later = first_and_next()
    print(f"[step time] first call {first * 1e3:.0f} us, later ones {later * 1e3:.0f} us", flush=True)
    assert first < 1.5 * later


def test_tiles_of_long_rows_hold_enough_rows(gpu, monkeypatch):
    """Two-step tiles with edges: a row of 120 or 124 cells taken whole leaves few rows to a tile, and a lattice of such
    rows took longer than one of 128 (FP32 256x128xnz: 94, 94 and 89 us a step; halved 85, 87 and 89)."""
    monkeypatch.setenv("PLBAMD_FUSED", "1")
    us = {}
    for nz in (120, 124, 128):
        with plb.Block3D(256, 128, nz, plb.D3Q19, plb.BGK(1.8), storage="f32") as lat:
            us[nz] = step_us(lat, 40)
    print(f"[step time] {us}", flush=True)
    assert max(us[120], us[124]) < 1.03 * us[128]
