"""A new porosity on a lattice that has run: it alone goes to the device (a
kernel out of the transfer's chunks in one block, a copy of every block's cells
otherwise), and adjoint calls share the buffer that the lattice keeps between
them. Everything must be what a fresh lattice gives, bit for bit."""
import os

import numpy as np
import pytest

from cases import Case, gpu_lattice, random_state, uneven_blocks, uniform
from oracle import oracle

import palabos_amd

pytestmark = pytest.mark.gpu

DTYPE = {"f64": np.float64, "f32": np.float32, "f16": np.uint16}


def make(case, blocks):
    if blocks is None:
        return gpu_lattice(case)
    lat = palabos_amd.Block3D(case.nx, case.ny, case.nz, palabos_amd.D3Q19, palabos_amd.RegularizedBGK(case.omega),
                              storage=case.storage, periodic=case.periodic, force=case.force, blocks=blocks,
                              keep_blocks=True)
    lat.setPorosity(case.alpha)
    return lat


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("tiling", ["single", "blocks"])
def test_new_porosity_between_steps(gpu, storage, tiling, pinned):
    shape = (13, 11, 24)
    case = Case(*shape, storage=storage, dynamics="rbgk", omega=1.6, periodic=(True, False, True),
                force=(1e-4, 0.0, 0.0), alpha=uniform(shape, 1))
    blocks = uneven_blocks(shape, [[5], [4], [10]]) if tiling == "blocks" else None
    f = oracle.to_storage(random_state(case, 5), storage)
    if not pinned:
        os.environ["PLBAMD_NO_PINNED"] = "1"
    try:
        lat = make(case, blocks)
        try:
            lat.setPopulations(f)
            for k, alpha in enumerate([case.alpha, uniform(shape, 2), None, 0.5 * uniform(shape, 3), uniform(shape, 4)]):
                print(f"[porosity] {storage} {tiling} {k}", flush=True)
                lat.setPorosity(alpha)
                lat.collideAndStream(3)
                case.alpha = np.zeros(shape) if alpha is None else alpha
                f, _ = oracle.run(case, f, 3)
                assert np.array_equal(lat.getPopulations(dtype=DTYPE[storage]), f)
        finally:
            lat.close()
    finally:
        os.environ.pop("PLBAMD_NO_PINNED", None)


@pytest.mark.parametrize("storage", ["f64", "f16"])
@pytest.mark.parametrize("tiling", ["single", "blocks"])
def test_repeated_gradients_share_the_buffer(gpu, storage, tiling):
    """Calls of different lengths, intervals and recording budgets in turn."""
    shape = (12, 10, 14)
    case = Case(*shape, storage=storage, dynamics="rbgk", omega=1.6, periodic=(True, False, True),
                force=(1e-4, 0.0, 0.0), alpha=0.5 * uniform(shape, 1))
    blocks = uneven_blocks(shape, [[6], [], [8]]) if tiling == "blocks" else None
    f0 = oracle.to_storage(random_state(case, 5) * 0.3, storage)

    def gradient(lat, alpha, T, K, budget):
        lat.setPorosity(alpha)
        lat.setPopulations(f0)
        lat.setAdjointRecordBytes(budget)
        J, ga, _, _ = lat.adjointGradient(T, K, 1, shape[0] - 2, 0.5, 1.0, weight_flux=2.0)
        return J, ga

    calls = [(1, 12, 4, -1), (2, 6, 2, 0), (3, 20, 4, 200000), (4, 4, 4, -1), (1, 12, 4, -1)]
    shared = make(case, blocks)
    try:
        got = [gradient(shared, 0.5 * uniform(shape, s), T, K, b) for s, T, K, b in calls]
    finally:
        shared.close()
    for (s, T, K, b), (J, ga) in zip(calls, got):
        lat = make(case, blocks)
        try:
            Jw, gw = gradient(lat, 0.5 * uniform(shape, s), T, K, b)
        finally:
            lat.close()
        assert J == Jw
        assert np.array_equal(ga, gw)
    assert np.array_equal(got[0][1], got[-1][1])
