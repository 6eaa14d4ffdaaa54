"""The reverse step at the extents where its launches change: rows one cell
around a wavefront's 64, row groups around four, every edge periodic or not
(also a single cell along an axis), planes in the bulk launch (few workgroups)
and in their own (more than 4096), adjoint states beyond 200 MB (nontemporal
accesses). J and the porosity gradient of 16 cells against the oracle's dual
numbers: rtol 1e-11 and 1e-8 (of FP64 sums in another order), atol 1e-13 of the
largest gradient."""
import numpy as np
import pytest

from cases import TAG_WALL, Case, channel_case, gpu_lattice, random_state, rest_state, uniform
from oracle import oracle

pytestmark = pytest.mark.gpu


def compare(case, f0, T, K, xin, xout, w_dp, w_drag, **kw):
    print(f"[adjoint] {case.shape} {case.dynamics} {case.periodic}", flush=True)
    pool = np.flatnonzero(case.alpha.ravel() > 0)
    seeds = np.sort(np.random.RandomState(1).choice(pool, 16, replace=pool.size < 16))
    lat = gpu_lattice(case)
    try:
        lat.setPopulations(f0)
        J, ga, gs, _ = lat.adjointGradient(T, K, xin, xout, w_dp, w_drag, weight_flux=kw.get("w_flux", 0.0),
                                           first_step=kw.get("first_step", 0))
    finally:
        lat.close()
    Jd, dJa, dJs = oracle.objective_dual(case, f0, T, xin, xout, w_dp, w_drag, seeds, **kw)
    assert J == pytest.approx(Jd, rel=1e-11)
    np.testing.assert_allclose(ga.ravel()[seeds], dJa, rtol=1e-8, atol=1e-13 * max(1e-3, np.abs(dJa).max()))
    return gs, dJs


@pytest.mark.parametrize("shape", [(3, 4, 63), (4, 5, 64), (3, 3, 65), (2, 7, 130), (5, 1, 20), (4, 6, 1)])
@pytest.mark.parametrize("dynamics,periodic,force", [
    ("bgk", (True, True, True), (1e-4, 0.0, 0.0)), ("rbgk", (False, True, False), (0.0, 0.0, 0.0)),
    ("rbgk", (True, False, True), (1e-4, -2e-5, 3e-5)), ("bgk", (False, False, False), (0.0, 0.0, 0.0)),
])
def test_extents(gpu, shape, dynamics, periodic, force):
    case = Case(*shape, dynamics=dynamics, omega=1.6, periodic=periodic, force=force,
                alpha=0.05 + 0.5 * uniform(shape, 4))
    compare(case, random_state(case, 6) * 0.3, 6, 2, 0, shape[0] - 1, 0.5, 1.0, w_flux=2.0, first_step=2)


@pytest.mark.parametrize("nz", [63, 66])
def test_link_walls_at_tile_edges(gpu, nz):
    case = Case(5, 9, nz, dynamics="rbgk", omega=1.6, periodic=(True, False, True), force=(1e-4, 0.0, 0.0))
    case.tags = np.zeros(case.shape, dtype=np.uint8)
    case.tags[2, 3:5, nz - 2:] = TAG_WALL
    case.tags[2, 3:5, :2] = TAG_WALL
    case.alpha = (0.05 + 0.4 * uniform(case.shape, 4)) * (case.tags == 0)
    compare(case, random_state(case, 6) * 0.3, 6, 2, 0, 4, 0.5, 1.0, w_flux=2.0, first_step=2)


@pytest.mark.parametrize("shape", [(12, 9, 64), (9, 8, 67), (2060, 5, 6)])
def test_planes_in_and_beside_the_bulk_launch(gpu, shape):
    case = channel_case(*shape, 1.6, 0.04)
    case.alpha = 0.05 + 0.5 * uniform(shape, 4)
    case.alpha[[0, -1]] = 0.0
    gs, dJs = compare(case, rest_state(case), 6, 2, 1, shape[0] - 2, 1.0, 1.0)
    assert gs[0] == pytest.approx(dJs, rel=1e-9)


def test_large_states(gpu):
    """96 x 84 x 84 FP64 cells: two adjoint states of 103 MB each."""
    case = Case(96, 84, 84, dynamics="bgk", omega=1.6, periodic=(True, True, True), force=(1e-4, 0.0, 0.0))
    case.alpha = 0.05 + 0.5 * uniform(case.shape, 4)
    compare(case, random_state(case, 6) * 0.3, 4, 2, 0, 95, 0.5, 1.0, w_flux=2.0)
