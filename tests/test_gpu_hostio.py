"""Cell data between host arrays and the device in chunks (csrc/hostio.h): the
chunks are whole x planes, rows of one plane or parts of one row, whatever fits
(256 KB at least, an eighth of the whole, 4 MB at most); every element must
arrive once. Lattices whose boxes take each of the three, sub-boxes that start
off the chunk edges, both layouts (after an even and an odd number of steps), and
the way without pinned memory."""
import os

import numpy as np
import pytest

import palabos_amd as plb
from cases import uniform

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (41, 20, 18), (2, 300, 130), (1, 3, 9001)]   # one cell; planes; rows; parts of a row


def boxes(shape):
    whole = tuple(v for n in shape for v in (0, n - 1))
    part = tuple(v for n in shape for v in (n // 3, n - 1 - n // 5))
    return [whole, part]


def lattice(shape):
    return plb.Block3D(*shape, plb.D3Q19, plb.BGK(1.7), storage="f64", periodic=True)


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("shape", SHAPES)
def test_populations_fields_and_moments(gpu, shape, pinned):
    if not pinned:
        os.environ["PLBAMD_NO_PINNED"] = "1"
    try:
        lat = lattice(shape)
        f = 0.02 * uniform(shape + (19,), 3)
        lat.setPopulations(f)
        assert np.array_equal(lat.getPopulations(), f)
        for x0, x1, y0, y1, z0, z1 in boxes(shape):
            box, cut = (x0, x1, y0, y1, z0, z1), np.s_[x0:x1 + 1, y0:y1 + 1, z0:z1 + 1]
            assert np.array_equal(lat.getPopulations(box), f[cut])
            g = 0.02 * uniform(f[cut].shape, 5)
            lat.setPopulations(g, box)
            f[cut] = g
            assert np.array_equal(lat.getPopulations(), f)
            rho, u = lat.macroscopic(box)
            c = plb_velocities()
            np.testing.assert_allclose(rho, 1.0 + f[cut].sum(-1), rtol=1e-13)
            np.testing.assert_allclose(u, (f[cut] @ c) / rho[..., None], rtol=1e-9, atol=1e-14)
            fields = lat.analysisFields(box)
            assert np.array_equal(fields[..., 0], rho) and np.array_equal(fields[..., 2:5], u)
        lat.collideAndStream(1)      # the swapped layout
        h = 0.02 * uniform(shape + (19,), 7)
        lat.setPopulations(h)
        assert np.array_equal(lat.getPopulations(), h)
        lat.computeRhoBarJ()
        rho_bar, j = lat.getRhoBarJ()
        lat.setRhoBarJ(2 * rho_bar, j - 1.0)
        again = lat.getRhoBarJ()
        assert np.array_equal(again[0], 2 * rho_bar) and np.array_equal(again[1], j - 1.0)
        r0, u0 = 1.0 + 0.01 * uniform(shape, 11), 0.02 * uniform(shape + (3,), 13)
        lat.initializeAtEquilibrium(r0, u0)
        rho, u = lat.macroscopic()
        np.testing.assert_allclose(rho, r0, rtol=1e-13)
        np.testing.assert_allclose(u, u0, rtol=1e-9, atol=1e-14)
        lat.close()
    finally:
        os.environ.pop("PLBAMD_NO_PINNED", None)


def plb_velocities():
    c = np.array([[0, 0, 0], [-1, 0, 0], [0, -1, 0], [0, 0, -1], [-1, -1, 0], [-1, 1, 0], [-1, 0, -1], [-1, 0, 1],
                  [0, -1, -1], [0, -1, 1]], dtype=np.float64)
    return np.concatenate([c, -c[1:]])
