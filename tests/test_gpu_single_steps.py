"""Single steps where the engine takes them on large lattices only: small ones are
taken two steps at a time or with statistics elsewhere in the tests. And two steps
at a time on a lattice whose reflections lie 2 to 4 GiB apart."""
import numpy as np
import pytest

import palabos_amd as plb
from cases import Case, gpu_lattice, random_state
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", ["0", "1", "2"])
@pytest.mark.parametrize("dynamics", ["bgk", "rbgk"])
@pytest.mark.parametrize("shape", [(5, 6, 128), (4, 3, 256), (3, 4, 514), (3, 3, 1030)])
@pytest.mark.parametrize("storage", ["f16", "bf16"])
def test_untagged_16_bit_pairs_without_statistics(gpu, monkeypatch, storage, shape, dynamics, policy):
    """The pair kernel of FP16 320^3 and 512^3 (periodic, no tags, no statistics): rows of one segment that wrap through
    LDS, and of several with halo words between; bit for bit the oracle's after even and odd steps."""
    monkeypatch.setenv("PLBAMD_FUSED", "0")
    monkeypatch.setenv("PLBAMD_CACHED_Z", policy)
    case = Case(*shape, storage=storage, dynamics=dynamics, omega=1.7, periodic=(True, True, True))
    f0 = oracle.to_storage(random_state(case, 17), storage)
    for steps in (5, 6):
        want, _ = oracle.run(case, f0, steps)
        lat = gpu_lattice(case)
        try:
            lat.toggleInternalStatistics(False)
            lat.setPopulations(f0)
            lat.collideAndStream(steps)
            assert lat.runInfo()["two_step_launches"] == 0
            got = lat.getPopulations(dtype=np.uint16)
        finally:
            lat.close()
        assert np.array_equal(got, want), f"{np.count_nonzero(got != want)} populations differ"


def test_two_steps_with_edges_over_4_gib_of_offsets(gpu, monkeypatch):
    """FP64, 300x300x360 with edges: a reflected population lies up to nine slots of 259 MB from its neighbour's, beyond
    2 GiB and within 4. Two steps at a time give the single steps' density and velocity bit for bit."""
    shape = (300, 300, 360)
    x, y, z = (np.arange(n, dtype=np.float64) for n in shape)
    u = np.empty(shape + (3,))
    u[..., 0] = 0.03 * np.sin(0.11 * x)[:, None, None] * np.cos(0.23 * y)[None, :, None]
    u[..., 1] = 0.02 * np.cos(0.17 * z)
    u[..., 2] = -0.03 * np.sin(0.19 * y)[None, :, None] * np.sin(0.07 * z)
    states = []
    for fused in ("0", "1"):
        monkeypatch.setenv("PLBAMD_FUSED", fused)
        with plb.Block3D(*shape, plb.D3Q19, plb.BGK(1.7), storage="f64") as lat:
            lat.toggleInternalStatistics(False)
            lat.initializeAtEquilibrium(1.0, u)
            lat.collideAndStream(6)
            assert lat.runInfo()["two_step_launches"] == (2 if fused == "1" else 0)
            states.append(lat.macroscopic())
    assert np.array_equal(states[0][0], states[1][0]) and np.array_equal(states[0][1], states[1][1])
    assert np.abs(states[0][1] - u).max() > 1e-4
