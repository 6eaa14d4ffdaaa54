"""The step kernels' cache policies (PLBAMD_CACHED_Z=0/1/2, read when a lattice
is created) and the launch that takes the special cells along with the bulk
rows (policy 2, 32- and 64-bit storage): single steps, bit for bit the
oracle's, on rows of one cell more and less than a wavefront and on few and
many special cells."""
import os

import numpy as np
import pytest

from cases import TAG_BB, Case, cavity_case, channel_case, gpu_lattice, random_state, sphere_tags
from oracle import oracle

pytestmark = pytest.mark.gpu

DTYPE = {"f64": np.float64, "f32": np.float32, "f16": np.uint16, "bf16": np.uint16}


def run(case, f0, n, policy, stats):
    env = {"PLBAMD_FUSED": "0", "PLBAMD_CACHED_Z": policy}
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        lat = gpu_lattice(case)
        try:
            lat.setPopulations(f0)
            lat.toggleInternalStatistics(stats)
            lat.collideAndStream(n)
            return lat.getPopulations(dtype=DTYPE[case.storage]), (lat.getStatistics() if stats else None)
        finally:
            lat.close()
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


def nodes_case(storage, nz):
    case = Case(7, 9, nz, storage=storage, omega=1.7, periodic=(True, False, nz % 2 == 0))
    case.tags = sphere_tags(case.shape, (3, 4, nz // 2), 2.4, TAG_BB)
    return case


@pytest.mark.parametrize("policy", ["0", "1", "2"])
@pytest.mark.parametrize("stats", [False, True])
@pytest.mark.parametrize("case", [
    *(cavity_case(11, 1.4, 0.05, storage=st, family="regularized", nz=nz) for st in ("f64", "f32", "f16")
      for nz in (3, 34, 65)),
    *(channel_case(12, 17, nz, 1.8, 0.05, storage=st, sphere=((5, 8, nz - 4), 3.3)) for st in ("f64", "f32", "f16")
      for nz in (20, 63, 130)),
    *(nodes_case(st, nz) for st in ("f64", "f32", "f16", "bf16") for nz in (64, 129)),
], ids=lambda c: f"{c.storage}-{c.nx}x{c.ny}x{c.nz}" if isinstance(c, Case) else None)
def test_policies(gpu, case, policy, stats):
    print(f"[policy] {case.shape} {case.storage} policy {policy} statistics {stats}", flush=True)
    f0 = oracle.to_storage(random_state(case, 4), case.storage)
    want, wst = oracle.run(case, f0, 5)
    got, gst = run(case, f0, 5, policy, stats)
    assert np.array_equal(got, want), f"{np.count_nonzero(got != want)} populations differ"
    if stats:
        np.testing.assert_allclose(gst["force"], wst["force"], rtol=1e-10, atol=1e-13)
        np.testing.assert_allclose(gst["avg_usqr"], wst["avg_usqr"], rtol=1e-10, atol=1e-15)
