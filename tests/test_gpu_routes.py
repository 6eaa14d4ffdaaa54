"""Which way a call runs (plbamd_get_run_info). The ways give the same
populations bit for bit, so the tests that compare results pass whichever was
taken: here the counts are compared."""
import pytest

import palabos_amd as plb
from cases import (TAG_BB, TAG_MEBB, TAG_NODYN, TAG_WALL, Case, cavity_case, channel_case, gpu_lattice,
                   sphere_tags)

pytestmark = pytest.mark.gpu


def pairs_of(calls, stats=False):
    """Launches of two steps in a sequence of calls: from an odd time on, as long as two steps are left that
    need not report statistics."""
    t = n = 0
    for steps in calls:
        end = t + steps
        while t < end:
            if t % 2 == 1 and end - t - int(stats) >= 2:
                t, n = t + 2, n + 1
            else:
                t += 1
    return n


def two_step_launches(lat, calls, stats=False):
    try:
        lat.toggleInternalStatistics(stats)
        for n in calls:
            lat.collideAndStream(n)
        return lat.runInfo()["two_step_launches"]
    finally:
        lat.close()


def cases_with_two_steps():
    nodes = Case(9, 17, 36, storage="f16", omega=1.8, periodic=(False, True, False))
    nodes.tags = sphere_tags(nodes.shape, (4, 8, 30), 4.2, TAG_BB)
    nodes.tags[2:4, 1:4, 0:3] = TAG_NODYN
    walls = Case(10, 16, 40, storage="f32", dynamics="rbgk", omega=1.7, periodic=(True, True, True), force=(1e-4, 0.0, 0.0))
    walls.tags = sphere_tags(walls.shape, (1, 14, 31), 4.5, TAG_WALL)
    return [Case(1, 1, 1, omega=1.7, periodic=(True, True, True)),
            Case(5, 14, 33, storage="bf16", omega=1.7, periodic=(True, True, True)),
            Case(7, 16, 34, storage="f32", dynamics="rbgk", omega=1.5, periodic=(False, False, False)),
            nodes, walls, channel_case(12, 17, 35, 1.8, 0.05, sphere=((5, 8, 31), 4.3))]


@pytest.mark.parametrize("stats", [False, True])
@pytest.mark.parametrize("calls", [[2], [3], [4], [5, 4], [1, 2, 3], [8]])
@pytest.mark.parametrize("case", cases_with_two_steps(), ids=lambda c: f"{c.storage}-{c.nx}x{c.ny}x{c.nz}")
def test_two_steps_are_launched(gpu, monkeypatch, case, calls, stats):
    monkeypatch.setenv("PLBAMD_FUSED", "1")
    assert two_step_launches(gpu_lattice(case), calls, stats) == pairs_of(calls, stats)


def test_two_steps_are_left_to_single_ones(gpu, monkeypatch):
    """Link walls beside nodes, boundary processors, several blocks, and PLBAMD_FUSED=0."""
    monkeypatch.setenv("PLBAMD_FUSED", "1")
    for tag in (TAG_BB, TAG_MEBB, TAG_NODYN):
        case = Case(8, 9, 33, omega=1.7, periodic=(True, True, True))
        case.tags = sphere_tags(case.shape, (4, 4, 10), 2.5, TAG_WALL)
        case.tags[1, 1, 30] = tag
        assert two_step_launches(gpu_lattice(case), [6]) == 0
    lat = plb.Block3D(8, 9, 10, plb.D3Q19, plb.BGK(1.7), storage="f64")
    lat.setVelocityConditionOnBlockBoundaries()
    assert two_step_launches(lat, [6]) == 0
    blocks = [(0, 7, 0, 8, 0, 9), (8, 15, 0, 8, 0, 9)]
    assert two_step_launches(plb.Block3D(16, 9, 10, plb.D3Q19, plb.BGK(1.7), storage="f64", periodic=True, blocks=blocks,
                                         keep_blocks=True), [6]) == 0
    monkeypatch.setenv("PLBAMD_FUSED", "0")
    assert two_step_launches(gpu_lattice(cavity_case(14, 1.4, 0.05)), [6]) == 0


def test_slots_are_padded_where_two_steps_are_taken(gpu):
    """16-bit lattices and several blocks, whose single steps the padding slows down, have none."""
    def stride(storage, **kw):
        with plb.Block3D(32, 24, 40, plb.D3Q19, plb.BGK(1.7), storage=storage, periodic=True, **kw) as lat:
            return lat.runInfo()["slot_stride"]
    cells = 32 * 24 * 40
    assert stride("f64") % 128 == stride("f32") % 128 == 64
    assert stride("f16") == stride("bf16") == cells
    blocks = [(0, 31, 0, 11, 0, 39), (0, 31, 12, 23, 0, 39)]
    assert stride("f32", blocks=blocks, keep_blocks=True) == 36 * 16 * 44   # two envelope layers a side


@pytest.mark.parametrize("storage, n, policy", [
    ("f64", 64, 2), ("f32", 64, 2), ("f16", 48, 2), ("f16", 56, 1), ("f16", 76, 1), ("f16", 84, 2), ("bf16", 48, 2),
    ("bf16", 56, 1), ("bf16", 76, 1), ("bf16", 84, 2), ("bf16", 65, 1)])
def test_cache_policy_of_small_lattices(gpu, storage, n, policy):
    """Ordinary loads (2) in the last-level cache, except 16-bit lattices of 6 to 19 MB, where they cost time."""
    with plb.Block3D(n, n, n, plb.D3Q19, plb.BGK(1.7), storage=storage, periodic=True) as lat:
        assert lat.runInfo()["cache_policy"] == policy


@pytest.mark.parametrize("storage, shape, kind, dynamics, force, taken", [
    # 16-bit, two cells per thread: FP16 BGK without edges, tags or force, 250,000 to 600,000 cells, rows up to 96
    ("f16", (32, 32, 32), "periodic", "bgk", False, False), ("f16", (72, 72, 72), "periodic", "bgk", False, True),
    ("f16", (96, 96, 96), "periodic", "bgk", False, False), ("f16", (44, 93, 128), "periodic", "bgk", False, False),
    ("f16", (72, 72, 72), "periodic", "rbgk", False, False), ("f16", (72, 72, 72), "periodic", "bgk", True, False),
    ("f16", (72, 72, 72), "box", "bgk", False, False), ("bf16", (72, 72, 72), "periodic", "bgk", False, False),
    # 16-bit, one cell per thread (odd nz)
    ("f16", (83, 85, 87), "periodic", "rbgk", False, False), ("f16", (101, 101, 101), "periodic", "rbgk", False, True),
    ("f16", (129, 131, 133), "box", "bgk", False, False), ("f16", (149, 151, 153), "box", "bgk", True, True),
    ("bf16", (101, 101, 101), "periodic", "bgk", False, False), ("bf16", (109, 109, 109), "periodic", "rbgk", False, True),
    ("bf16", (149, 151, 153), "box", "bgk", False, False), ("bf16", (191, 203, 197), "box", "bgk", False, True),
    # FP32: regularized BGK or a force from 430,000 cells on; with edges and rows of broken lines from 900,000
    ("f32", (68, 75, 62), "periodic", "rbgk", False, False), ("f32", (68, 75, 62), "periodic", "bgk", False, True),
    ("f32", (60, 88, 64), "periodic", "bgk", True, False), ("f32", (80, 80, 80), "periodic", "rbgk", False, True),
    ("f32", (97, 99, 101), "box", "rbgk", True, True), ("f32", (83, 85, 87), "box", "rbgk", False, False),
    ("f32", (83, 85, 87), "box", "bgk", False, True),
    # FP64 with edges or tags: with a force not between 800,000 and 2,300,000 cells (whole lines; the cache otherwise)
    ("f64", (80, 80, 80), "box", "rbgk", True, True), ("f64", (112, 112, 112), "box", "rbgk", True, False),
    ("f64", (128, 128, 128), "walls", "rbgk", True, False), ("f64", (112, 112, 112), "box", "rbgk", False, True),
    ("f64", (112, 112, 112), "periodic", "rbgk", True, True), ("f64", (97, 99, 101), "box", "rbgk", True, False),
    ("f64", (129, 131, 133), "walls", "rbgk", True, True), ("f64", (160, 160, 160), "walls", "rbgk", True, True)])
def test_two_steps_where_they_are_the_faster_way(gpu, monkeypatch, storage, shape, kind, dynamics, force, taken):
    monkeypatch.delenv("PLBAMD_FUSED", raising=False)
    dyn = plb.BGK(1.7) if dynamics == "bgk" else plb.RegularizedBGK(1.7)
    lat = plb.Block3D(*shape, plb.D3Q19, dyn, storage=storage, periodic=kind != "box", force=(1e-5, 0.0, 0.0) if force else None)
    if kind == "walls":
        lat.defineDynamics((5, 5, 5, 5, 5, 5), plb.WallLink)
    assert two_step_launches(lat, [5]) == (2 if taken else 0)
