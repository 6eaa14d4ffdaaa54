"""The work that a user of this framework has it do, as timed cases.

Every case goes through the public Python interface (palabos_amd.Block3D) and
returns what the program goes on with: the populations or the density and
velocity of every cell after the steps, forces, gradients. The solvers are
iterated many times between two read-outs in practice, so a pass advances the
lattice by many steps and then reads the whole result once.

Lattices of more than about 40 million cells are left out (the 512^3 of the
headline benchmark among them): their read-out alone is many gigabytes; from
256^3 cells on the populations no longer fit any cache of the device.

work() counts, as is usual for these solvers, every step as one read and one
write of the populations (19 values each per cell), what the step reads besides
them once, and the read-out.

exact() restates the path in plain torch, in 64 bits.
"""
import math

import numpy as np
import torch

import palabos_amd as plb
from palabos_amd import setups

SIZE = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # The reference's regression case (jlabos doctest): velocity conditions on every
        # face, edge and corner of a small box, 30 steps. The smallest calls: a step is
        # half a dozen launches over few cells.
        {"name": "cavity_all_boundaries_f64", "kind": "doctest", "nx": 20, "ny": 31, "nz": 42, "storage": "f64",
         "steps": 30},
        # Lid-driven cavity, the 64^3 validation configuration, with the statistics read
        # every 20 steps as a convergence monitor does.
        {"name": "cavity64_monitored_f64", "kind": "cavity", "nx": 64, "ny": 64, "nz": 64, "storage": "f64",
         "steps": 400, "every": 20},
        # Decaying vortex in a periodic box, the headline workload, in the three storage
        # types: FP64 at a power of two, FP32 at ragged extents, 16 bits at the largest size.
        {"name": "taylor_green_256_f64", "kind": "taylor_green", "nx": 256, "ny": 256, "nz": 256, "storage": "f64",
         "dynamics": "bgk", "steps": 400},
        {"name": "taylor_green_ragged_f32", "kind": "taylor_green", "nx": 191, "ny": 203, "nz": 197, "storage": "f32",
         "dynamics": "rbgk", "steps": 801},
        {"name": "taylor_green_320_f16", "kind": "taylor_green", "nx": 320, "ny": 320, "nz": 320, "storage": "f16",
         "dynamics": "bgk", "steps": 360},
        # Channel flow past a sphere, the drag configuration: Zou-He inlet and outlet,
        # momentum-exchange sphere, force sampled every 10 steps.
        {"name": "sphere_channel_f32", "kind": "sphere", "nx": 256, "ny": 128, "nz": 128, "radius": 16.0,
         "storage": "f32", "steps": 800, "every": 10},
        # Permeability of a medium of link-wall spheres, driven by a body force, 16-bit storage.
        {"name": "porous_spheres_f16", "kind": "porous", "nx": 256, "ny": 160, "nz": 128, "spheres": 80,
         "storage": "f16", "steps": 800},
        # A lattice kept as the caller's uneven blocks (as a distributed set-up hands it over),
        # bounce-back obstacle, walls, body force; odd extents.
        {"name": "kept_blocks_f32", "kind": "blocks", "nx": 129, "ny": 97, "nz": 75, "storage": "f32",
         "dynamics": "bgk", "steps": 200},
        # One design iteration of the Brinkman channel: new porosity, forward and reverse sweep.
        {"name": "adjoint_channel_f64", "kind": "adjoint_channel", "nx": 128, "ny": 64, "nz": 64, "storage": "f64",
         "steps": 200, "checkpoint": 50},
        # The permeability gradient of a smooth sphere medium, 16-bit forward, regularized BGK.
        {"name": "adjoint_porous_f16", "kind": "adjoint_porous", "nx": 192, "ny": 128, "nz": 128, "spheres": 40,
         "storage": "f16", "steps": 40, "checkpoint": 20},
        # A coupling code around the step: moments out, changed by the program, back in,
        # collide with them (multiphase and free-surface models).
        {"name": "external_coupling_f64", "kind": "external", "nx": 64, "ny": 60, "nz": 72, "storage": "f64",
         "steps": 10},
        # The co-processor seam: populations handed over, a few steps, populations taken back.
        {"name": "coprocessor_round_trip_f64", "kind": "round_trip", "nx": 100, "ny": 88, "nz": 70, "storage": "f64",
         "dynamics": "bgk", "steps": 15},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# cells * steps of the listed case of a kind: a drawn case costs no more
_BUDGET = {"doctest": 30 * 26040, "cavity": 400 * 64 ** 3, "taylor_green": 300 * 256 ** 3, "sphere": 600 * 256 * 128 * 128,
           "porous": 600 * 256 * 160 * 128, "blocks": 200 * 129 * 97 * 75, "adjoint_channel": 200 * 128 * 64 * 64,
           "adjoint_porous": 40 * 192 * 128 * 128, "external": 10 * 64 * 60 * 72, "round_trip": 15 * 100 * 88 * 70}


def draw(rng):
    # the step in its three settings (box, channel, medium) oftener than the work around it
    kind = rng.choice(sorted(_BUDGET) + ["taylor_green"] * 3 + ["sphere", "porous", "cavity"])
    d = lambda lo, hi: _log_int(rng, lo, hi)  # noqa: E731
    c = {"kind": kind}
    if kind == "doctest":
        c.update(nx=d(12, 30), ny=d(12, 31), nz=d(12, 42), storage=rng.choice(["f64", "f32"]), steps=30)
    elif kind == "cavity":
        c.update(nx=d(20, 72), ny=d(20, 72), nz=d(20, 72), storage=rng.choice(["f64", "f32"]), every=rng.choice([10, 20, 25]))
    elif kind == "taylor_green":
        n = d(32, 250)
        c.update(nx=n, ny=max(16, n + rng.randint(-6, 6)), nz=max(16, n + rng.randint(-6, 6)),
                 storage=rng.choice(["f64", "f32", "f16", "bf16"]), dynamics=rng.choice(["bgk", "rbgk"]))
    elif kind == "sphere":
        c.update(nx=d(64, 250), ny=d(32, 126), nz=d(32, 126), storage=rng.choice(["f64", "f32", "f16"]),
                 every=rng.choice([5, 10, 20]))
        c["radius"] = round(min(c["ny"], c["nz"]) / 8.0, 2)
    elif kind == "porous":
        c.update(nx=d(64, 250), ny=d(48, 156), nz=2 * d(24, 62), storage=rng.choice(["f16", "f16", "f32", "f64"]))
        c["spheres"] = max(4, c["nx"] * c["ny"] * c["nz"] // 66000)
    elif kind == "blocks":
        c.update(nx=d(40, 128), ny=d(32, 96), nz=d(32, 75), storage=rng.choice(["f64", "f32", "f16"]),
                 dynamics=rng.choice(["bgk", "rbgk"]))
    elif kind == "adjoint_channel":
        c.update(nx=d(40, 126), ny=d(24, 63), nz=d(24, 63), storage="f64", checkpoint=rng.choice([20, 40, 50]))
    elif kind == "adjoint_porous":
        c.update(nx=d(64, 190), ny=d(48, 126), nz=2 * d(24, 62), storage=rng.choice(["f16", "f64"]), checkpoint=20)
        c["spheres"] = max(4, c["nx"] * c["ny"] * c["nz"] // 80000)
    elif kind == "external":
        c.update(nx=d(20, 62), ny=d(20, 58), nz=d(20, 70), storage=rng.choice(["f64", "f32"]))
    else:
        c.update(nx=d(24, 98), ny=d(24, 86), nz=d(24, 68), storage=rng.choice(["f64", "f32"]),
                 dynamics=rng.choice(["bgk", "rbgk"]))
    if "steps" not in c:
        cells = c["nx"] * c["ny"] * c["nz"]
        most = {"cavity": 600, "taylor_green": 600, "sphere": 600, "porous": 600, "blocks": 400, "adjoint_channel": 240,
                "adjoint_porous": 80, "external": 20, "round_trip": 30}[kind]
        n = max(4, min(most, int(_BUDGET[kind] * rng.uniform(0.5, 1.0) / cells)))
        c["steps"] = n // 2 * 2 if kind.startswith("adjoint") else n
    return c


def work(case):
    cells = case["nx"] * case["ny"] * case["nz"]
    size, kind, steps = SIZE[case["storage"]], case["kind"], case["steps"]
    step_bytes, step_flops = 38 * size, 240 if case.get("dynamics", "bgk") == "bgk" else 360
    if kind in ("adjoint_channel", "adjoint_porous"):
        # forward step with the pre-collision moments written; reverse step: the adjoint state
        # read and written, moments and porosity read, gradient read and written
        a = 8 if case["storage"] == "f64" else 4
        step_bytes += 4 * a + a + 38 * a + 4 * a + a + 2 * a
        step_flops += 420
    elif kind == "external":
        # moments written, read out, set and read by the step
        step_bytes += 19 * size + 4 * size + 2 * (4 * size + 32) + 4 * size
    out = {"doctest": 19 * 8, "cavity": 19 * 8, "taylor_green": 32, "sphere": 32, "porous": 32, "blocks": 19 * 4,
           "adjoint_channel": 2 * 19 * 8 + 16, "adjoint_porous": 16, "external": 19 * 8,
           "round_trip": 2 * 19 * size}[kind]
    return {"bytes": float(cells * (steps * step_bytes + out)), "flops": float(cells * steps * step_flops)}


# ---------------------------------------------------------------------------
# Inputs, from the seed alone (the same for the framework and for exact())

def _omega(kind):
    return {"doctest": 1.0, "cavity": 1.4, "taylor_green": 1.8, "porous": 1.7, "blocks": 1.6, "adjoint_channel": 1.6,
            "adjoint_porous": 1.7, "external": 1.5, "round_trip": 1.8}[kind]


def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _waves(shape, seed, u0):
    """A velocity field of periodic Taylor-Green waves with amplitudes and phases from the seed."""
    rng = np.random.RandomState(seed % (1 << 31))
    p = rng.uniform(0.0, 2.0 * np.pi, 3)
    a = u0 * rng.uniform(0.7, 1.0)
    w = [2.0 * np.pi / n * np.arange(n) + q for n, q in zip(shape, p)]
    sx, cx = np.sin(w[0])[:, None, None], np.cos(w[0])[:, None, None]
    sy, cy = np.sin(w[1])[None, :, None], np.cos(w[1])[None, :, None]
    cz = np.cos(w[2])[None, None, :]
    u = np.empty(tuple(shape) + (3,))
    u[..., 0] = a * (sx * cy) * cz
    u[..., 1] = -a * (cx * sy) * cz
    u[..., 2] = 0.1 * a * (sx * sy)
    return u


def _box_solid(shape, seed):
    """An off-centre box obstacle."""
    rng = np.random.RandomState(seed % (1 << 31))
    m = np.zeros(shape, dtype=bool)
    lo = [int(n * rng.uniform(0.3, 0.4)) for n in shape]
    m[tuple(slice(q, q + max(2, n // 5)) for q, n in zip(lo, shape))] = True
    return m


def _slab_walls(shape):
    m = np.zeros(shape, dtype=bool)
    m[:, :, 0] = m[:, :, -1] = True
    return m


def _sphere_solid(case, seed):
    rng = np.random.RandomState(seed % (1 << 31))
    nx, ny, nz = _shape(case)
    centre = (nx / 4.0 + rng.uniform(-2, 2), ny / 2.0 + rng.uniform(-2, 2), nz / 2.0 + rng.uniform(-2, 2))
    return setups.sphere_mask((nx, ny, nz), centre, case["radius"])


def _medium(case, seed):
    shape = _shape(case)
    hi = min(14.0, min(shape) / 8.0)
    return setups.random_spheres(shape, case["spheres"], (0.45 * hi, hi), seed % (1 << 31), periodic=(True, False, False))


def _smooth_spheres(case, seed):
    from palabos_amd.studies import brinkman_spheres
    centres, radii = _medium(case, seed)
    return brinkman_spheres(_shape(case), centres, radii)[0]


def _blob_porosity(case, seed):
    a = setups.brinkman_blobs(_shape(case), n_blobs=12, seed=seed % (1 << 31))
    a[0] = a[-1] = 0.0
    return a


def _inlet(case, seed, u_max):
    rng = np.random.RandomState(seed % (1 << 31))
    prof = setups.poiseuille_profile(case["ny"], case["nz"], u_max * rng.uniform(0.8, 1.0))
    v = np.zeros((prof.size, 3))
    v[:, 0] = prof.reshape(-1)
    return v


def _uneven_cuts(shape):
    return [[n * 3 // 7] if a else [n // 4, n * 5 // 8] for a, n in enumerate(shape)]


_W = np.array([1 / 3.] + ([1 / 18.] * 3 + [1 / 36.] * 6) * 2)
_C = np.array([[0, 0, 0], [-1, 0, 0], [0, -1, 0], [0, 0, -1], [-1, -1, 0], [-1, 1, 0], [-1, 0, -1], [-1, 0, 1],
               [0, -1, -1], [0, -1, 1]])
_C = np.concatenate([_C, -_C[1:]])


def _populations(shape, seed, u0=0.03):
    """Populations a host program hands over: equilibrium of a wave field plus a smooth non-equilibrium part."""
    u = _waves(shape, seed, u0)
    cu = u @ _C.T.astype(np.float64)
    u2 = (u * u).sum(-1)[..., None]
    return np.ascontiguousarray(_W * (3.0 * cu + 4.5 * cu * cu - 1.5 * u2) * (1.0 + 0.05 * cu))


def _dynamics(case):
    w = _omega(case["kind"])
    return plb.RegularizedBGK(w) if case.get("dynamics", "bgk") == "rbgk" else plb.BGK(w)


def _sphere_omega(case):
    return 1.0 / (3.0 * 0.05 * 2.0 * case["radius"] / 100.0 + 0.5)


_FORCE = 1e-5
_COUPLING = 2e-6


def prepare(case, seed):
    kind, shape, st = case["kind"], _shape(case), case["storage"]
    nx, ny, nz = shape
    s = {"case": case}
    if kind == "doctest":
        rng = np.random.RandomState(seed % (1 << 31))
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.BGK(_omega(kind)), storage=st)
        lat.setVelocityConditionOnBlockBoundaries("regularized", wrapped=True)
        u = np.array([0.02 * rng.uniform(0.7, 1.0), 0.005 * rng.uniform(-1.0, 1.0), 0.0])
        lat.setBoundaryVelocityIn((1, nx - 2, 1, ny - 2, nz - 1, nz - 1), u)
    elif kind == "cavity":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.BGK(_omega(kind)), storage=st)
        lid = lat.addVelocityBoundary(2, 1, (1, nx - 2, 1, ny - 2, nz - 1, nz - 1))
        lat.setBoundaryVelocity(lid, _lid(seed))
    elif kind == "taylor_green":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, _dynamics(case), storage=st, periodic=True)
        lat.initializeAtEquilibrium(1.0, _waves(shape, seed, 0.04))
        lat.toggleInternalStatistics(False)
    elif kind == "sphere":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.BGK(_sphere_omega(case)), storage=st)
        lat.defineDynamics(_sphere_solid(case, seed), plb.MomentumExchangeBounceBack)
        p = lat.addVelocityBoundary(0, -1, (0, 0, 1, ny - 2, 1, nz - 2))
        lat.setBoundaryVelocity(p, _inlet(case, seed, 0.05))
        p = lat.addPressureBoundary(0, 1, (nx - 1, nx - 1, 1, ny - 2, 1, nz - 2))
        lat.setBoundaryDensity(p, 1.0)
    elif kind == "porous":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.RegularizedBGK(_omega(kind)), storage=st,
                          periodic=(True, False, False), force=(_FORCE, 0.0, 0.0))
        lat.defineDynamics(setups.spheres_mask(shape, *_medium(case, seed), periodic=(True, False, False)), plb.WallLink)
        lat.toggleInternalStatistics(False)
    elif kind == "blocks":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, _dynamics(case), storage=st, periodic=(True, False, False),
                          force=(_FORCE, 0.0, 0.0), blocks=setups.tile_blocks(shape, _uneven_cuts(shape)),
                          keep_blocks=True)
        lat.defineDynamics(_box_solid(shape, seed), plb.BounceBack)
        lat.initializeAtEquilibrium(1.0, _waves(shape, seed, 0.02))
        lat.toggleInternalStatistics(False)
    elif kind == "adjoint_channel":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.BGK(_omega(kind)), storage=st)
        p = lat.addVelocityBoundary(0, -1, (0, 0, 1, ny - 2, 1, nz - 2))
        lat.setBoundaryVelocity(p, _inlet(case, seed, 0.04))
        p = lat.addPressureBoundary(0, 1, (nx - 1, nx - 1, 1, ny - 2, 1, nz - 2))
        lat.setBoundaryDensity(p, 1.0)
        s["alpha"] = _blob_porosity(case, seed)
        s["rest"] = np.zeros(shape + (19,))
    elif kind == "adjoint_porous":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.RegularizedBGK(_omega(kind)), storage=st,
                          periodic=(True, False, False), force=(_FORCE, 0.0, 0.0))
        s["alpha"] = _smooth_spheres(case, seed)
    elif kind == "external":
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, plb.BGK(_omega(kind)), storage=st, periodic=True)
        lat.defineDynamics(_slab_walls(shape), plb.BounceBack)
        lat.initializeAtEquilibrium(1.0, _waves(shape, seed, 0.02))
    else:
        lat = plb.Block3D(nx, ny, nz, plb.D3Q19, _dynamics(case), storage=st, periodic=(True, True, False))
        lat.toggleInternalStatistics(False)
        s["f"] = _populations(shape, seed).astype(np.float64 if st == "f64" else np.float32)
    s["lattice"] = lat
    return s


def _lid(seed):
    return np.array([0.05 * np.random.RandomState(seed % (1 << 31)).uniform(0.7, 1.0), 0.01, 0.0])


def run(state):
    case, lat = state["case"], state["lattice"]
    kind, steps = case["kind"], case["steps"]
    dtype = np.float64 if case["storage"] == "f64" else np.float32
    if kind == "doctest":
        lat.initialize()
        lat.collideAndStream(steps)
        return {"density": lat.averageDensity(), "energy": lat.averageEnergy(), "f": lat.getPopulations(dtype=dtype)}
    if kind in ("cavity", "sphere"):
        series = []
        for k in range(0, steps, case["every"]):
            lat.collideAndStream(min(case["every"], steps - k))
            st = lat.getStatistics()
            series.append([st["avg_rhobar"], st["avg_usqr"]] if kind == "cavity" else list(st["force"]))
        if kind == "cavity":
            return {"series": np.array(series), "f": lat.getPopulations(dtype=dtype)}
        rho, u = lat.macroscopic()
        return {"force": np.array(series), "rho": rho, "u": u}
    if kind in ("taylor_green", "porous"):
        lat.collideAndStream(steps)
        rho, u = lat.macroscopic()
        return {"rho": rho, "u": u}
    if kind == "adjoint_channel":
        lat.setPorosity(state["alpha"])
        lat.setPopulations(state["rest"])
        J, ga, gs, _ = lat.adjointGradient(steps, case["checkpoint"], 1, case["nx"] - 2, 1.0, 1.0)
        return {"J": J, "grad_alpha": ga, "grad_scale": gs, "f": lat.getPopulations()}
    if kind == "adjoint_porous":
        lat.setPorosity(state["alpha"])
        lat.initializeAtEquilibrium(1.0, (0.0, 0.0, 0.0))
        J, ga, _, _ = lat.adjointGradient(steps, case["checkpoint"], 0, 0, 0.0, 0.0, weight_flux=1.0,
                                          first_step=steps // 2)
        return {"J": J, "grad_alpha": ga}
    if kind == "external":
        for _ in range(steps):
            lat.computeRhoBarJ()
            rho_bar, j = lat.getRhoBarJ()
            j[..., 0] += _COUPLING * (1.0 + rho_bar)
            lat.setRhoBarJ(rho_bar, j)
            lat.externalCollideAndStream(1)
        return {"f": lat.getPopulations()}
    if kind == "round_trip":
        lat.setPopulations(state["f"])
    lat.collideAndStream(steps)
    return {"f": lat.getPopulations(dtype=dtype)}


# ---------------------------------------------------------------------------
# The same in plain torch, in 64 bits

def _opp(i):
    return 0 if i == 0 else (i + 9 if i <= 9 else i - 9)


class _Torch:
    def __init__(self, case, periodic, omega, dynamics="bgk", force=0.0, links=None, bounce=None):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.shape, self.omega, self.dynamics, self.force = _shape(case), omega, dynamics, force
        self.c = torch.tensor(_C, dtype=torch.float64, device=self.dev)
        self.w = torch.tensor(_W, dtype=torch.float64, device=self.dev)
        self.links = None if links is None else torch.tensor(links, device=self.dev)
        self.bounce = None if bounce is None else torch.tensor(bounce, device=self.dev)
        self.swap = [_opp(i) for i in range(19)]
        self.mask = []
        idx = [torch.arange(n, device=self.dev) for n in self.shape]
        for i in range(19):
            m = None
            for a in range(3):
                if _C[i, a] and not periodic[a]:
                    src = idx[a] - int(_C[i, a])
                    out = ((src < 0) | (src >= self.shape[a])).view([-1 if b == a else 1 for b in range(3)])
                    m = out if m is None else m | out
            if i and self.links is not None:
                wall = torch.roll(self.links, _C[i].tolist(), (0, 1, 2))
                m = wall if m is None else m | wall
            self.mask.append(m)

    def t(self, a):
        return torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)

    def wide(self, v):
        return v.view(-1, 1, 1, 1)

    def moments(self, f):
        return f.sum(0), torch.tensordot(self.c.T, f, 1)

    def equilibrium(self, rho_bar, j):
        cj = torch.tensordot(self.c, j, 1)
        return self.wide(self.w) * (rho_bar + 3 * cj + (4.5 * cj * cj - 1.5 * (j * j).sum(0)) / (1 + rho_bar))

    def collide(self, f, alpha=None, given=None):
        rho_bar, j = self.moments(f) if given is None else given
        rho, w = 1 + rho_bar, self.omega
        u = j / rho
        if self.force:
            u = torch.cat([u[:1] + 0.5 * self.force, u[1:]])
        if alpha is not None:
            u = (1 - alpha) * u
        eq = self.equilibrium(rho_bar, rho * u)
        if self.dynamics == "bgk":
            g = (1 - w) * f + w * eq
        else:
            g = eq
            for a in range(3):
                for b in range(a, 3):
                    cc = self.c[:, a] * self.c[:, b]
                    pi = torch.tensordot(cc, f, 1) - j[a] * j[b] / rho - (rho_bar / 3 if a == b else 0.0)
                    q = (cc - (1 / 3. if a == b else 0.0)) * (4.5 * self.w * (1 if a == b else 2))
                    g = g + (1 - w) * self.wide(q) * pi
        if self.force:
            cx, cu = self.wide(self.c[:, 0]), torch.tensordot(self.c, u, 1)
            g = g + (1 - w / 2) * self.wide(self.w) * self.force * (3 * (cx - u[0]) + 9 * cu * cx)
        if self.bounce is not None:
            g = torch.where(self.bounce, f[self.swap], g)
        return g

    def stream(self, g):
        out = []
        for i in range(19):
            v = torch.roll(g[i], _C[i].tolist(), (0, 1, 2)) if i else g[0]
            out.append(v if self.mask[i] is None else torch.where(self.mask[i], g[_opp(i)], v))
        return torch.stack(out)

    def plane(self, f, direction, side, u=None):
        """rhoBar and j of the cells of a Zou-He plane (u imposed, or rho = 1)."""
        on, out = [i for i in range(19) if _C[i, direction] == 0], [i for i in range(19) if _C[i, direction] == side]
        total = 2 * f[out].sum(0) + f[on].sum(0)
        if u is not None:
            rho_bar = (total - side * u[direction]) / (1 + side * u[direction])
            return rho_bar, (1 + rho_bar) * u
        j = torch.zeros((3,) + tuple(total.shape), dtype=f.dtype, device=f.device)
        j[direction] = side * total
        return torch.zeros_like(total), j

    def zou_he(self, f, direction, side, u=None):
        rho_bar, j = self.plane(f, direction, side, u)
        eq = self.equilibrium(rho_bar, j)
        g = list(f)
        for n in range(19):
            if _C[n, direction] == side:
                g[_opp(n)] = f[n] - eq[n] + eq[_opp(n)]
        excess = (j - torch.tensordot(self.c.T, torch.stack(g), 1)) / 4
        for n in range(19):
            p = _opp(n)
            if _C[n, direction] == side and abs(_C[p]).sum() > 1:
                for a in ((direction + 1) % 3, (direction + 2) % 3):
                    g[p] = g[p] + int(_C[p, a]) * excess[a]
        return torch.stack(g)

    def host(self, f):
        return np.ascontiguousarray(f.permute(1, 2, 3, 0).cpu().numpy())

    def read(self, f, rho_bar=None, u=None):
        r, j = self.moments(f)
        v = j / (1 + r)
        if self.force:
            v[0] += 0.5 * self.force
        if self.links is not None:
            r, v = torch.where(self.links, 0.0, r), torch.where(self.links, 0.0, v)
        return r, v


def _exact_channel(case, seed, T):
    nx, ny, nz = _shape(case)
    u = T.t(_inlet(case, seed, 0.05 if case["kind"] == "sphere" else 0.04)).T.reshape(3, 1, ny - 2, nz - 2)
    lo, hi = (slice(None), slice(0, 1), slice(1, -1), slice(1, -1)), (slice(None), slice(nx - 1, nx), slice(1, -1), slice(1, -1))

    def complete(f, scale=1.0):
        f = f.clone()
        a, b = T.zou_he(f[lo].clone(), 0, -1, scale * u), T.zou_he(f[hi].clone(), 0, 1)
        f[lo], f[hi] = a, b
        return f
    return u, lo, hi, complete


def _objective(case, T, f, alpha):
    rho_bar, j = T.moments(f)
    if case["kind"] == "adjoint_porous":
        return j[0].mean()
    return (rho_bar[1].mean() - rho_bar[case["nx"] - 2].mean()) / 3 + T.omega * (alpha * j[0]).sum()


def _exact_adjoint(case, seed):
    channel = case["kind"] == "adjoint_channel"
    if channel:
        T = _Torch(case, (False,) * 3, _omega(case["kind"]))
        complete = _exact_channel(case, seed, T)[3]
        alpha, t0 = T.t(_blob_porosity(case, seed)), 0
    else:
        T = _Torch(case, (True, False, False), _omega(case["kind"]), "rbgk", _FORCE)
        alpha, t0 = T.t(_smooth_spheres(case, seed)), case["steps"] // 2
    step = lambda f, a, s: T.stream(T.collide(complete(f, s) if channel else f, a))  # noqa: E731
    states = [torch.zeros((19,) + T.shape, dtype=torch.float64, device=T.dev)]
    weight = 1.0 / (case["steps"] - t0)
    J = 0.0
    with torch.no_grad():
        for t in range(case["steps"]):
            states.append(step(states[-1], alpha, 1.0))
            if t + 1 > t0:
                J += weight * float(_objective(case, T, states[-1], alpha))
    last = T.host(states[-1]) if channel else None
    lam, ga, gs = torch.zeros_like(states[0]), torch.zeros_like(alpha), 0.0
    for t in range(case["steps"], -1, -1):
        f = states.pop().requires_grad_()
        a, s = alpha.clone().requires_grad_(), torch.ones((), dtype=torch.float64, device=T.dev, requires_grad=True)
        total = weight * _objective(case, T, f, a) if t > t0 else 0.0 * (f.sum() + a.sum())
        if t < case["steps"]:
            total = total + (lam * step(f, a, s)).sum()
        g = torch.autograd.grad(total, (f, a, s), allow_unused=True)
        lam = g[0]
        ga += 0.0 if g[1] is None else g[1]
        gs += 0.0 if g[2] is None else float(g[2])
    if channel:   # the porosity is zero on the planes, and no gradient is reported there
        ga[[0, -1], 1:-1, 1:-1] = 0.0
    out = {"J": J, "grad_alpha": ga.cpu().numpy()}
    return dict(out, grad_scale=np.array([gs, 0.0]), f=last) if channel else out


def exact(case, seed):
    kind, steps, shape = case["kind"], case["steps"], _shape(case)
    cells = shape[0] * shape[1] * shape[2]
    if kind == "doctest" or cells * steps * (1.8 if case.get("dynamics") == "rbgk" else 1.0) > 1.2e10:
        return None   # the finite-difference edges are not restated here; or too long
    if kind.startswith("adjoint"):
        return _exact_adjoint(case, seed)
    with torch.no_grad():
        return _exact_forward(case, seed, kind, steps, shape)


def _exact_forward(case, seed, kind, steps, shape):
    dyn = case.get("dynamics", "bgk")
    if kind == "cavity":
        T = _Torch(case, (False,) * 3, _omega(kind))
        lid = (slice(None), slice(1, -1), slice(1, -1), slice(shape[2] - 1, shape[2]))
        u = T.t(_lid(seed)).view(3, 1, 1, 1)
        f, series = torch.zeros((19,) + shape, dtype=torch.float64, device=T.dev), []
        for k in range(steps):
            f = f.clone()
            f[lid] = T.zou_he(f[lid].clone(), 2, 1, u)
            if (k + 1) % case["every"] == 0 or k + 1 == steps:
                r, j = T.moments(f)
                series.append([float(r.mean()), float((j * j).sum(0).div((1 + r) ** 2).mean())])
            f = T.stream(T.collide(f))
        return {"series": np.array(series), "f": T.host(f)}
    if kind == "sphere":
        solid = _sphere_solid(case, seed)
        T = _Torch(case, (False,) * 3, _sphere_omega(case), bounce=solid)
        u, lo, hi, complete = _exact_channel(case, seed, T)
        f, series = torch.zeros((19,) + shape, dtype=torch.float64, device=T.dev), []
        m = T.bounce
        fluid = [m & ~torch.roll(m, (-_C[i]).tolist(), (0, 1, 2)) for i in range(19)]
        for k in range(steps):
            if (k + 1) % case["every"] == 0 or k + 1 == steps:
                through = torch.stack([(f[_opp(i)] * fluid[i]).sum() for i in range(19)])
                series.append((-2.0 * (T.c * through[:, None]).sum(0)).tolist())
            f = T.stream(T.collide(complete(f)))
        rho, v = T.read(f)
        rho[lo[1:]], v[lo] = T.plane(f[lo], 0, -1, u)[0], u.expand_as(v[lo])
        rho[hi[1:]], v[hi] = 0.0, T.plane(f[hi], 0, 1)[1]
        rho, v = torch.where(m, 0.0, rho), torch.where(m, 0.0, v)
        return {"force": np.array(series), "rho": 1 + rho.cpu().numpy(), "u": np.moveaxis(v.cpu().numpy(), 0, -1)}
    if kind == "external":
        T = _Torch(case, (True,) * 3, _omega(kind), bounce=_slab_walls(shape))
    elif kind == "porous":
        links = setups.spheres_mask(shape, *_medium(case, seed), periodic=(True, False, False))
        T = _Torch(case, (True, False, False), _omega(kind), "rbgk", _FORCE, links=links)
    elif kind == "blocks":
        T = _Torch(case, (True, False, False), _omega(kind), dyn, _FORCE, bounce=_box_solid(shape, seed))
    elif kind == "round_trip":
        T = _Torch(case, (True, True, False), _omega(kind), dyn)
    else:
        T = _Torch(case, (True,) * 3, _omega(kind), dyn)
    if kind == "round_trip":
        f = T.t(np.moveaxis(_populations(shape, seed), -1, 0))
    elif kind == "porous":
        f = torch.zeros((19,) + shape, dtype=torch.float64, device=T.dev)
    else:
        u = T.t(np.moveaxis(_waves(shape, seed, 0.04 if kind == "taylor_green" else 0.02), -1, 0))
        f = T.equilibrium(torch.zeros_like(u[0]), u)
    for _ in range(steps):
        given = None
        if kind == "external":
            rho_bar, j = T.moments(f)
            rho_bar, j = torch.where(T.bounce, 0.0, rho_bar), torch.where(T.bounce, 0.0, j)
            j[0] += _COUPLING * (1 + rho_bar)
            given = rho_bar, j
        f = T.stream(T.collide(f, given=given))
    if kind in ("taylor_green", "porous"):
        rho, v = T.read(f)
        return {"rho": 1 + rho.cpu().numpy(), "u": np.moveaxis(v.cpu().numpy(), 0, -1)}
    return {"f": T.host(f)}
