"""Odd steps over the cells of several blocks in memory order (the default there)
and row by row (PLBAMD_LINEAR_ODD=0, read when a lattice is created): bit for bit
the oracle's populations, statistics included. Cuts along every axis and along one,
rows shorter and longer than a wavefront, walls, link walls, nodes, force, porosity."""
import os

import numpy as np
import pytest

import palabos_amd
from cases import TAG_BB, TAG_WALL, Case, random_state, sphere_tags, uneven_blocks, uniform
from oracle import oracle

pytestmark = pytest.mark.gpu

DTYPE = {"f64": np.float64, "f32": np.float32}


@pytest.mark.parametrize("linear", ["1", "0"])
@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("shape,cuts", [((13, 12, 31), [[4], [5], [12]]), ((9, 14, 70), [[], [6], []]),
                                        ((8, 9, 141), [[], [], [66]]), ((17, 7, 10), [[5, 11], [], []])])
@pytest.mark.parametrize("kind", ["walls", "periodic", "links"])
def test_blocks_odd_steps(gpu, linear, storage, shape, cuts, kind):
    case = Case(*shape, storage=storage, dynamics="rbgk" if kind == "periodic" else "bgk", omega=1.7,
                periodic={"walls": (False,) * 3, "periodic": (True,) * 3, "links": (True, False, True)}[kind])
    if kind != "walls":
        case.force = (1e-4, -2e-5, 3e-5)
        case.alpha = 0.4 * uniform(shape, 2)
    centre = (shape[0] // 2, shape[1] // 2, shape[2] - 3)
    case.tags = None if kind == "periodic" else sphere_tags(shape, centre, 2.6, TAG_BB if kind == "walls" else TAG_WALL)
    old = os.environ.get("PLBAMD_LINEAR_ODD")
    os.environ["PLBAMD_LINEAR_ODD"] = linear
    try:
        print(f"[linear odd] {shape} {storage} {kind} {linear}", flush=True)
        dyn = palabos_amd.BGK(case.omega) if case.dynamics == "bgk" else palabos_amd.RegularizedBGK(case.omega)
        lat = palabos_amd.Block3D(*shape, palabos_amd.D3Q19, dyn, storage=storage, periodic=case.periodic,
                                  force=case.force, blocks=uneven_blocks(shape, cuts), keep_blocks=True)
        try:
            if case.tags is not None:
                lat.defineDynamics(case.tags != 0, palabos_amd.BounceBack if kind == "walls" else palabos_amd.WallLink)
            if case.alpha is not None:
                lat.setPorosity(case.alpha)
            f0 = oracle.to_storage(random_state(case, 4), storage)
            lat.setPopulations(f0)
            lat.collideAndStream(6)
            got, gst = lat.getPopulations(dtype=DTYPE[storage]), lat.getStatistics()
        finally:
            lat.close()
    finally:
        if old is None:
            del os.environ["PLBAMD_LINEAR_ODD"]
        else:
            os.environ["PLBAMD_LINEAR_ODD"] = old
    want, wst = oracle.run(case, f0, 6)
    if kind == "links":
        got[case.tags == TAG_WALL] = 0
        want[case.tags == TAG_WALL] = 0
    assert np.array_equal(got, want), f"{np.count_nonzero(got != want)} populations differ"
    np.testing.assert_allclose(gst["avg_usqr"], wst["avg_usqr"], rtol=1e-10, atol=1e-15)
