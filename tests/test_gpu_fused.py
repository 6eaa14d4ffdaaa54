"""Two steps per launch (csrc/fused.h), which lattices of a few million cells
take, forced on small ones through PLBAMD_FUSED=1 (read by every call): the
populations and the statistics must be the oracle's bit for bit. Extents
around the tile edges (one cell, a tile less one, a tile more one, rows of
several tiles), the shortest sequences of steps that contain a fused pair,
either start parity, every storage, both dynamics, a force with porosity,
non-periodic edges, bounce-back and inert nodes, link walls, and boundary
planes with a momentum-exchange sphere."""
import os

import numpy as np
import pytest

from cases import (TAG_BB, TAG_MEBB, TAG_NODYN, TAG_WALL, Case, cavity_case, channel_case, gpu_lattice, random_state,
                   sphere_tags, uniform)
from oracle import oracle

pytestmark = pytest.mark.gpu

DTYPE = {"f64": np.float64, "f32": np.float32, "f16": np.uint16, "bf16": np.uint16}


def fused_run(case, f0, calls, stats=False):
    old = os.environ.get("PLBAMD_FUSED")
    os.environ["PLBAMD_FUSED"] = "1"
    try:
        lat = gpu_lattice(case)
        try:
            lat.setPopulations(f0)
            lat.toggleInternalStatistics(stats)
            for n in calls:
                lat.collideAndStream(n)
            return lat.getPopulations(dtype=DTYPE[case.storage]), (lat.getStatistics() if stats else None)
        finally:
            lat.close()
    finally:
        if old is None:
            del os.environ["PLBAMD_FUSED"]
        else:
            os.environ["PLBAMD_FUSED"] = old


def check(case, calls, seed=3, skip=None, stats=False):
    print(f"[fused] {case.shape} {case.storage} {case.dynamics} {case.periodic} {calls}", flush=True)
    f0 = oracle.to_storage(random_state(case, seed), case.storage)
    want, wst = oracle.run(case, f0, sum(calls))
    got, gst = fused_run(case, f0, calls, stats)
    if skip is not None:
        assert np.array_equal(got[skip], f0[skip])   # link-wall solid keeps its values
        want, got = want.copy(), got.copy()
        want[skip] = 0
        got[skip] = 0
    assert np.array_equal(got, want), f"{np.count_nonzero(got != want)} populations differ"
    if stats:
        np.testing.assert_allclose(gst["force"], wst["force"], rtol=1e-10, atol=1e-13)
        np.testing.assert_allclose(gst["avg_usqr"], wst["avg_usqr"], rtol=1e-10, atol=1e-15)


@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 2), (4, 13, 32), (5, 14, 33), (2, 27, 131), (33, 3, 50)])
def test_periodic_extents(gpu, storage, shape):
    check(Case(*shape, storage=storage, omega=1.7, periodic=(True, True, True)), [6])


@pytest.mark.parametrize("calls", [[3], [4], [5, 4], [1, 2, 3], [8]])
def test_step_sequences(gpu, calls):
    check(Case(6, 15, 35, storage="f32", dynamics="rbgk", omega=1.6, periodic=(True, False, True)), calls)


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dynamics", ["bgk", "rbgk"])
@pytest.mark.parametrize("periodic", [(False, False, False), (True, False, True), (False, True, True), (True, True, False)])
def test_edges_force_and_porosity(gpu, storage, dynamics, periodic):
    shape = (7, 16, 34)
    check(Case(*shape, storage=storage, dynamics=dynamics, omega=1.5, periodic=periodic, force=(1e-4, -2e-5, 3e-5),
               alpha=0.5 + 0.5 * uniform(shape, 9)), [7])


@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("periodic", [(True, True, True), (False, True, False)])
def test_nodes(gpu, storage, periodic):
    case = Case(9, 17, 36, storage=storage, omega=1.8, periodic=periodic)
    tags = sphere_tags(case.shape, (4, 8, 30), 4.2, TAG_BB)
    tags[2:4, 1:4, 0:3] = TAG_NODYN
    case.tags = tags
    check(case, [6])


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("periodic", [(True, True, True), (True, False, False)])
def test_link_walls(gpu, storage, periodic):
    case = Case(10, 16, 40, storage=storage, dynamics="rbgk", omega=1.7, periodic=periodic, force=(1e-4, 0.0, 0.0))
    case.tags = sphere_tags(case.shape, (1, 14, 31), 4.5, TAG_WALL)
    case.tags[6, 3, 5] = TAG_WALL
    check(case, [6], skip=case.tags == TAG_WALL)


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
def test_planes_and_momentum_exchange(gpu, storage):
    check(channel_case(12, 17, 35, 1.8, 0.05, storage=storage, sphere=((5, 8, 31), 4.3)), [7, 4], stats=True)
    check(cavity_case(14, 1.4, 0.05, storage=storage, family="regularized", nz=34), [8], stats=True)
    check(channel_case(9, 16, 20, 1.6, 0.04, storage=storage, sphere=((4, 8, 9), 3.3), sphere_tag=TAG_BB), [5])


def test_walls_beside_nodes_keep_single_steps(gpu):
    """Link walls next to bounce-back and momentum-exchange nodes are not taken two steps at a time."""
    case = Case(8, 9, 33, omega=1.7, periodic=(True, True, True))
    case.tags = sphere_tags(case.shape, (4, 4, 10), 2.5, TAG_WALL)
    case.tags[sphere_tags(case.shape, (4, 4, 20), 2.5, 1) != 0] = TAG_BB
    case.tags[1, 1, 30] = TAG_MEBB
    solid = case.tags == TAG_WALL
    f0 = random_state(case, 5)
    want, _ = oracle.run(case, f0, 6)
    got, _ = fused_run(case, f0, [6])
    assert np.array_equal(got[~solid], want[~solid])


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("periodic", [(True, True, True), (False, False, False)])
@pytest.mark.parametrize("shape", [(5, 70, 150), (40, 34, 66), (3, 65, 128)])
def test_several_tiles_of_1024_threads(gpu, storage, periodic, shape):
    check(Case(*shape, storage=storage, omega=1.7, periodic=periodic), [6])
