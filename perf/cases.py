"""Performance cases of the SPH framework, each through its public entry points.

A case is a dict of plain values; `kind` says which entry points it runs:

  steps      whole time steps of the C++ HeterogeneousSimulator (lib.Simulator:
             fused step replayed as a graph, the defaults), from a particle
             state that is loaded into it before every pass
  launchers  one time step through the reference's own launchers (gCalcHashKey,
             sort, cells, gCalcMassDensity, gSPHCalculateForces, gSPHIntegrate)
             with arrays that the caller owns, as a program ported from the
             reference calls them
  layers     the density pass and the force + integration pass alone, on a
             fluid that is already sorted (fg_sph_density_nbr,
             fg_sph_forces_integrate_nbr)
  coupled    one step of a fluid with a floating torus and a static cylinder
             through the C launchers, up to the per-body force sums
  sort       the key/value sort alone (fg_sort_pairs_ws)
  ensemble   a whole run of many independent scenes (lib.BatchSimulator) from
             host arrays to host arrays
  mesh       winding numbers of a mesh on its sampling lattice
             (fg_mesh_winding_lattice)

Fluids are blocks of nx x ny x nz particles at half the kernel radius, as the
dam-break configurations have them, disturbed as in a running simulation:
every position is off its lattice point by up to a fifth of the spacing, and
the velocities are a smooth swirl with noise.  `order` is "lattice" (particles
numbered layer by layer, as an emitter numbers them: early in a run) or
"mixed" (any order: late in a run, when the fluid has been stirred).
"""
import ctypes as C
import math

import numpy as np
import torch

from fluidgrid_amd import abi, lib, mesh, scenes

DEV = "cuda"
F = np.float32


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # The reference application's scene as it ships: hashed keys, about
        # 24,000 particles, one step a frame.
        dict(name="frame_app_24k", kind="steps", keys="xor", nx=41, ny=28, nz=21, precision="fp32", steps=1,
             order="lattice"),
        # The smallest dam break: a few steps a frame, where launches and latency count.
        dict(name="frames_dam_16k", kind="steps", keys="linear", nx=32, ny=16, nz=32, precision="fp32", steps=4,
             order="lattice"),
        # The ordinary dam break of 1,048,576 particles.
        dict(name="steps_dam_1m", kind="steps", keys="linear", nx=128, ny=64, nz=128, precision="fp32", steps=4,
             order="lattice"),
        # Odd sizes, late in a run: the particles' numbers no longer follow the grid.
        dict(name="step_late_4m", kind="steps", keys="linear", nx=203, ny=101, nz=203, precision="fp32", steps=1,
             order="mixed"),
        # The largest configuration's fluid, 33,554,432 particles.
        dict(name="step_dam_33m", kind="steps", keys="linear", nx=512, ny=256, nz=256, precision="fp32", steps=1,
             order="lattice"),
        # The mixed-precision density form.
        dict(name="step_mixed_2m", kind="steps", keys="linear", nx=161, ny=81, nz=161, precision="mixed", steps=1,
             order="lattice"),
        # A program ported from the reference, launcher by launcher, in a mid-size fluid.
        dict(name="launchers_250k", kind="launchers", keys="linear", nx=63, ny=63, nz=63, order="lattice"),
        # The two neighbour passes alone, in a ragged fluid.
        dict(name="layers_2m", kind="layers", nx=160, ny=83, nz=159, order="mixed"),
        # The headline coupled workload's stages: 1,048,576 particles and a torus of about 20,000
        # spheres, here floating in the fluid beside a static cylinder.
        dict(name="coupled_1m", kind="coupled", nx=128, ny=64, nz=128, order="lattice", torus=0.15),
        # The sort alone, at a size that is no multiple of anything.
        dict(name="sort_3m", kind="sort", n=3000017, bits=24),
        # An ensemble with bodies, from the scenes' initial arrays to the final ones.
        dict(name="ensemble_128", kind="ensemble", scenes=128, low=4096, high=65536, steps=96, bodies=True),
        # Sampling a mesh of 20,000 triangles.
        dict(name="mesh_20k", kind="mesh", nu=125, nv=80, across=96),
    ]


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "launchers", "layers", "coupled", "sort", "ensemble", "mesh"])

    def log_between(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def block(lo, hi):
        """Lattice of about the drawn number of particles, flat to tall."""
        n, flat, deep = log_between(lo, hi), rng.uniform(0.4, 1.2), rng.uniform(0.6, 1.5)
        nx = max(6, round((n / (flat * deep)) ** (1 / 3)) + rng.randint(-1, 1))
        nz = max(6, round(nx * deep))
        return dict(nx=nx, ny=max(4, round(n / (nx * nz))), nz=nz)

    order = rng.choice(["lattice", "mixed"])
    if kind == "steps":
        keys = rng.choice(["linear", "linear", "linear", "xor"])
        size = block(8e3, 1.2e5) if keys == "xor" else block(6e3, 1.2e7)
        precision = rng.choice(["fp32", "fp32", "mixed"]) if keys == "linear" else "fp32"
        n = size["nx"] * size["ny"] * size["nz"]
        return dict(kind=kind, keys=keys, precision=precision, steps=rng.randint(1, 4) if n < 2e6 else 1, order=order,
                    **size)
    if kind == "launchers":
        keys = rng.choice(["linear", "xor"])
        return dict(kind=kind, keys=keys, order=order, **(block(8e3, 1.2e5) if keys == "xor" else block(1e4, 2e6)))
    if kind == "layers":
        return dict(kind=kind, order=order, **block(1.5e4, 6e6))
    if kind == "coupled":
        return dict(kind=kind, order=order, torus=round(rng.uniform(0.08, 0.18), 4), **block(1e5, 3e6))
    if kind == "sort":
        return dict(kind=kind, n=int(log_between(2e3, 3e7)) | 1, bits=rng.randint(14, 28))
    if kind == "ensemble":
        return dict(kind=kind, scenes=rng.randint(9, 100), low=4096, high=rng.randint(8192, 65536),
                    steps=rng.randint(20, 120), bodies=rng.random() < 0.5)
    return dict(kind=kind, nu=rng.randint(30, 130), nv=rng.randint(20, 80), across=rng.randint(24, 110))


def work(case):
    kind = case["kind"]
    if kind == "sort":
        return {"bytes": 16.0 * case["n"], "flops": 0.0}
    if kind == "mesh":
        _, dims, tris = _mesh_size(case)
        points = dims[0] * dims[1] * dims[2]
        return {"bytes": 4.0 * points + 12.0 * tris + 6.0 * tris, "flops": 60.0 * points * tris}
    # A particle of a fluid at rest has 33 others within its kernel radius: about 12 operations a
    # pair for the density and 40 for the forces.
    if kind == "ensemble":
        n = sum(s.n for s in _ensemble(case).scenes)
        return {"bytes": 64.0 * n * case["steps"], "flops": 33.0 * 52.0 * n * case["steps"]}
    n = case["nx"] * case["ny"] * case["nz"]
    steps = case.get("steps", 1)
    # position and velocity in and out, keys, ids and density out
    return {"bytes": (64.0 + 16.0) * n * steps, "flops": 33.0 * 52.0 * n * steps}


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------

def _scene(case):
    """The scene's parameters as plain numbers (FP32 values where the
    parameter blocks hold FP32)."""
    lat = (case["nx"], case["ny"], case["nz"])
    if case["keys"] == "xor":
        # AppMain.cpp:84-123: mass and kernel radius from the particle count.
        s = float(F(0.009))
        mass = F(F(131072.0) / F(24000.0)) * F(0.0002)
        dist = np.power(F(mass / F(1000.0)), F(F(1.0) / F(3.0)))
        spacing = float(F(F(dist * F(0.87)) / F(s)))
        h = float(F(F(F(2.0) * dist) * F(0.87)))
        cell = float(F(F(h) / F(s)))
        vmin = (-20.0, -20.0, -20.0)
        vmax = tuple(max(a, v + spacing * (m + 2)) for a, v, m in zip((20.0, 85.0, 40.0), vmin, lat))
        sc = dict(origin=vmin, spacing=spacing, h=h, s=s, cell=cell, vmin=vmin, vmax=vmax, dims=(64, 64, 64),
                  dt=float(F(0.004)), g=float(F(-9.8)), mass=float(mass), k=1.5, mu=1.0, point=spacing)
    else:
        # the dam-break configurations: h so that the block's longest side is 0.64 m
        h = float(F(1.28 / max(lat)))
        spacing = 0.5 * h
        dims = tuple(int(math.ceil(1.2 * m)) + 3 for m in (lat[0] / 2 * 1.3, lat[1] / 2 * 1.6, lat[2] / 2))
        vmax = tuple(float(F(d * h)) for d in dims)
        sc = dict(origin=(spacing, spacing, spacing), spacing=spacing, h=h, s=1.0, cell=h, vmin=(0.0, 0.0, 0.0),
                  vmax=vmax, dims=dims, dt=float(F(0.015 * h)), g=float(F(-9.81)),
                  mass=float(F(1000.0 * spacing ** 3)), k=3.0, mu=3.5, point=float(F(0.5 * 0.25 * h)))
    h = sc["h"]
    pi = float(F(3.14159265))
    sc.update(n=lat[0] * lat[1] * lat[2], lattice=lat, rho0=1000.0, limit=600.0, mode=case["keys"],
              buckets=sc["dims"][0] * sc["dims"][1] * sc["dims"][2],
              poly6=float(F(315.0 / (float(F(64.0 * pi)) * h ** 9))), spiky=float(F(-(45.0 / (pi * h ** 6)))),
              visc=float(F(45.0 / (pi * h ** 6))))
    return sc


def _blocks(sc):
    """The scene's parameter blocks."""
    cp = abi.CommonFluidParams()
    cp.cell_size = abi.f3(sc["cell"], sc["cell"], sc["cell"])
    cp.bucket_size = abi.i3(*sc["dims"])
    cp.keyBits = scenes.key_bits(sc["buckets"])
    cp.kernel_radius = sc["h"]
    cp.kernel_radius_squared = float(F(F(sc["h"]) * F(sc["h"])))
    cp.pointRadius, cp.pointScale, cp.velocity_limit = sc["point"], 1.0, sc["limit"]
    cp.volume_min, cp.volume_max = abi.f3(*sc["vmin"]), abi.f3(*sc["vmax"])
    cp.global_external_force = abi.f3(0.0, sc["g"], 0.0)
    cp.simulation_scale, cp.deltaTimeIntegration = sc["s"], sc["dt"]
    cp.fluid_to_srb_relation = abi.i3(1, 1, 1)
    fp = abi.FluidParams()
    fp.mass, fp.restDensity, fp.viscosity, fp.gasConstant = sc["mass"], sc["rho0"], sc["mu"], sc["k"]
    fp.particle_radius, fp.max_particles = sc["point"], sc["n"]
    kc = abi.KernelsCache()
    kc.kPoly6, kc.kSpikyGradient, kc.kViscosityLaplacian = sc["poly6"], sc["spiky"], sc["visc"]
    return cp, fp, kc


def _fluid(sc, order, seed):
    """Positions and velocities, float32 [n, 4] on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    nx, ny, nz = sc["lattice"]
    n, d = sc["n"], sc["spacing"]
    i = torch.arange(n, device=DEV)
    at = torch.stack([i % nx, i // (nx * nz), (i // nx) % nz], 1).float()
    del i
    u = torch.rand(n, 3, generator=g, device=DEV)
    pos = torch.ones(n, 4, device=DEV)
    pos[:, :3] = (at + 0.4 * u - 0.2) * d + torch.tensor(sc["origin"], device=DEV)
    del u
    vel = torch.zeros(n, 4, device=DEV)
    turn = 6.2831853 / (d * max(sc["lattice"]))
    q = pos[:, :3] * turn
    vel[:, 0] = 0.5 * torch.sin(q[:, 1]) * torch.cos(q[:, 2])
    vel[:, 1] = -0.3 * torch.sin(q[:, 0])
    vel[:, 2] = 0.4 * torch.cos(q[:, 0] + q[:, 1])
    vel[:, :3] += 0.05 * torch.randn(n, 3, generator=g, device=DEV)
    if order == "mixed":
        p = torch.randperm(n, generator=g, device=DEV)
        pos, vel = pos[p].contiguous(), vel[p].contiguous()
    return pos, vel


def _mesh_size(case):
    """(spacing, lattice dimensions, triangles) of a torus mesh of major radius 0.3 and minor 0.1."""
    spacing = 0.8 / case["across"]
    dims = (case["across"] + 2, int(0.2 / spacing) + 3, case["across"] + 2)
    return spacing, dims, 2 * case["nu"] * case["nv"]


_ENSEMBLES = {}


def _ensemble(case):
    key = (case["scenes"], case["low"], case["high"], case["bodies"])
    if key not in _ENSEMBLES:
        _ENSEMBLES.clear()
        _ENSEMBLES[key] = scenes.ensemble(case["scenes"], n_range=(case["low"], case["high"]), bodies=case["bodies"])
    return _ENSEMBLES[key]


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------

class _Raw:
    """A device array that the library owns, for torch.as_tensor."""

    def __init__(self, ptr, shape, kind):
        self.__cuda_array_interface__ = dict(shape=shape, typestr=kind, data=(ptr, False), version=2)


# The simulator is one per process by its API: a program keeps one and steps
# it; the states of one case share it and load their particles into it.
_KEPT = {}


def _drop():
    if _KEPT:
        _KEPT.pop("sim").close()
        _KEPT.clear()


def _simulator(case, sc):
    key = (sc["mode"], sc["lattice"], case["precision"])
    if _KEPT.get("key") != key:
        _drop()
        cp, fp, kc = _blocks(sc)
        zero = np.zeros((sc["n"], 4), np.float32)
        scene = scenes.Scene("case", zero, zero, fp, cp, kc, abi.KEY_REF_XOR if sc["mode"] == "xor" else abi.KEY_LINEAR,
                             1)
        sim = lib.Simulator(scene, precision=abi.PRECISION_MIXED if case["precision"] == "mixed" else
                            abi.PRECISION_FP32)
        b, n = sim.buffers, sc["n"]
        _KEPT.update(key=key, sim=sim, out=dict(
            pos=torch.as_tensor(_Raw(b.position, (n, 4), "<f4"), device=DEV),
            vel=torch.as_tensor(_Raw(b.velocity, (n, 4), "<f4"), device=DEV),
            rho_p=torch.as_tensor(_Raw(b.densityPressure, (n, 2), "<f4"), device=DEV),
            ids=torch.as_tensor(_Raw(b.particleId, (n,), "<i4"), device=DEV)))
    return _KEPT


def _params(sc):
    cp, _, kc = _blocks(sc)
    lib.init_params(cp, kc, abi.KEY_REF_XOR if sc["mode"] == "xor" else abi.KEY_LINEAR)


def _i32(*shape):
    return torch.empty(*shape, dtype=torch.int32, device=DEV)


def _f32(*shape):
    return torch.zeros(*shape, device=DEV)


class _Grid:
    """A caller's own arrays for one fluid's grid."""

    def __init__(self, sc):
        n, nb = sc["n"], sc["buckets"]
        self.bits = scenes.key_bits(nb)
        self.keys, self.ids = _i32(n), _i32(n)
        self.start, self.end = _i32(nb), _i32(nb)
        self.spos, self.svel, self.rho = _f32(n, 4), _f32(n, 4), _f32(n, 2)
        self.ws_bytes = lib.load().fg_sort_workspace_size(n, self.bits)
        self.ws = torch.empty(self.ws_bytes, dtype=torch.uint8, device=DEV)


def _sort_into_cells(sc, g, pos, vel):
    """Keys, stable sort, cells and the sorted copies."""
    L, n, cs = lib.load(), sc["n"], abi.f3(sc["cell"], sc["cell"], sc["cell"])
    L.gCalcHashKey(g.keys.data_ptr(), g.ids.data_ptr(), pos.data_ptr(), n, sc["buckets"], cs)
    L.fg_sort_pairs_ws(g.keys.data_ptr(), g.ids.data_ptr(), n, g.bits, g.ws.data_ptr(), g.ws_bytes, 0)
    L.gFindCellOffsetOrderingPosVel(g.start.data_ptr(), g.end.data_ptr(), g.keys.data_ptr(), g.ids.data_ptr(),
                                    pos.data_ptr(), g.spos.data_ptr(), vel.data_ptr(), g.svel.data_ptr(), n,
                                    sc["buckets"])


def _bodies(case, sc):
    """A torus half in the fluid and a static cylinder standing in it, as
    plain arrays and numbers."""
    h, d = sc["h"], sc["spacing"]
    span = [m * d for m in sc["lattice"]]
    R = case["torus"]
    torus = scenes.torus_spheres(R, R / 3.0, d) + np.array([0.5 * span[0], span[1], 0.5 * span[2]])
    post = scenes.cylinder_spheres(0.05, 0.5 * span[1], d) + np.array([0.15 * span[0], d, 0.2 * span[2]])
    return dict(torus=np.concatenate([torus, np.zeros((len(torus), 1))], 1).astype(np.float32),
                post=np.concatenate([post, np.zeros((len(post), 1))], 1).astype(np.float32),
                centre=np.array([0.5 * span[0], span[1], 0.5 * span[2]], np.float32),
                radius=float(F(0.5 * h)), fluid_radius=float(F(2.0 * sc["point"])),
                cell=float(F(max(0.75 * h + 0.003, h + 0.001) * 1.01)), buckets=64 ** 3, spring=-2000.0, damping=-50.0)


def _body_grid(b, start, end, spheres, bounds, vel, count):
    g = abi.BodyGrid()
    g.orderedSpheres, g.gridStart, g.gridEnd, g.bounds = (t.data_ptr() for t in (spheres, start, end, bounds))
    g.bodyVelocities = vel.data_ptr() if vel is not None else None
    g.cellSize = abi.f3(b["cell"], b["cell"], b["cell"])
    g.numBuckets, g.relation, g.numSpheres = b["buckets"], abi.i3(1, 1, 1), count
    g.numBodies = 1 if vel is not None else 0
    g.fluidRadius, g.sphereRadius, g.kSpring, g.kDamping = b["fluid_radius"], b["radius"], b["spring"], b["damping"]
    return g


class _Spheres:
    """The arrays of one body's sphere grid."""

    def __init__(self, b, rel):
        L, m = lib.load(), len(rel)
        self.m = m
        self.rel = torch.from_numpy(rel).to(DEV)
        self.world, self.sorted = _f32(m, 4), _f32(m, 4)
        self.keys, self.ids = _i32(m), _i32(m)
        self.start, self.end = _i32(b["buckets"]), _i32(b["buckets"])
        self.bounds = _f32(2, 4)
        self.bits = scenes.key_bits(b["buckets"])
        self.ws_bytes = L.fg_sort_workspace_size(m, self.bits)
        self.ws = torch.empty(self.ws_bytes, dtype=torch.uint8, device=DEV)

    def build(self, b, cm, orient):
        """World transform, keys, sort, cells and bounds."""
        L = lib.load()
        L.gCalcHashKeyWithOffset(self.keys.data_ptr(), self.ids.data_ptr(), cm.data_ptr(), orient.data_ptr(),
                                 self.rel.data_ptr(), self.world.data_ptr(), self.m,
                                 abi.f3(b["cell"], b["cell"], b["cell"]), b["buckets"])
        L.fg_sort_pairs_ws(self.keys.data_ptr(), self.ids.data_ptr(), self.m, self.bits, self.ws.data_ptr(),
                           self.ws_bytes, 1)
        L.gFindCellOffsetOrderingPos(self.start.data_ptr(), self.end.data_ptr(), self.keys.data_ptr(),
                                     self.ids.data_ptr(), self.world.data_ptr(), self.sorted.data_ptr(), self.m,
                                     b["buckets"])
        margin = (b["fluid_radius"] + b["radius"] + 0.003) * 1.01
        L.fg_sphere_bounds(self.world.data_ptr(), self.m, margin, self.bounds.data_ptr())


def _full(case):
    """A case with the fields that its kind leaves at their usual values."""
    return dict(dict(keys="linear", precision="fp32", order="lattice"), **case)


def prepare(case, seed):
    case = _full(case)
    kind = case["kind"]
    if kind == "steps":
        sc = _scene(case)
        kept = _simulator(case, sc)
        pos, vel = _fluid(sc, case["order"], seed)
        return dict(kind=kind, steps=case["steps"], pos=pos, vel=vel, bytes=16 * sc["n"], kept=kept)
    _drop()
    if kind in ("launchers", "layers", "coupled"):
        sc = _scene(case)
        _params(sc)
        g = _Grid(sc)
        pos, vel = _fluid(sc, case["order"], seed)
        st = dict(kind=kind, sc=sc, g=g, pos=pos, vel=vel, pos_out=pos.clone(), vel_out=vel.clone())
        if kind != "launchers":
            st["nbr"] = torch.empty(lib.load().fg_neighbor_mask_bytes(sc["n"]), dtype=torch.uint8, device=DEV)
        if kind == "layers":
            _sort_into_cells(sc, g, pos, vel)
        if kind == "coupled":
            b = _bodies(case, sc)
            torus, post = b["torus"].copy(), b["post"]
            torus[:, :3] -= b["centre"]
            st.update(b=b, torus=_Spheres(b, torus), post=_Spheres(b, post),
                      cm=torch.tensor([[*b["centre"], 0.0]], device=DEV),
                      bvel=torch.tensor([[0.1, -0.4, 0.05, 0.0]], device=DEV),
                      orient=torch.tensor([[0.0, 0.0, 0.0, 1.0]], device=DEV),
                      offsets=torch.tensor([0, len(torus)], dtype=torch.int32, device=DEV),
                      pf=_f32(len(torus), 4), pt=_f32(len(torus), 4),
                      sums=torch.zeros(2, 1, 4, dtype=torch.float64, device=DEV))
            st["post"].build(b, torch.zeros(1, 4, device=DEV), st["orient"])  # static: built once
        return st
    g = torch.Generator(device=DEV).manual_seed(seed)
    if kind == "sort":
        n = case["n"]
        # cell keys of a fluid: runs of about eight equal keys, in no order
        keys = torch.randint(0, 1 << case["bits"], ((n + 7) // 8,), generator=g, device=DEV)
        keys = keys[torch.randint(0, len(keys), (n,), generator=g, device=DEV)].int()
        ws = lib.load().fg_sort_workspace_size(n, case["bits"])
        return dict(kind=kind, n=n, bits=case["bits"], keys=keys, vals=torch.arange(n, dtype=torch.int32, device=DEV),
                    k=_i32(n), v=_i32(n), ws=torch.empty(ws, dtype=torch.uint8, device=DEV), ws_bytes=ws)
    if kind == "mesh":
        v, t = _mesh(case, seed)
        spacing, dims, _ = _mesh_size(case)
        return dict(kind=kind, v=torch.from_numpy(v).to(DEV), t=torch.from_numpy(t.astype(np.int32)).to(DEV),
                    dims=dims, spacing=spacing, out=_f32(dims[0] * dims[1] * dims[2]))
    ens = _ensemble(case)
    rng = np.random.default_rng(seed)
    moved = []
    for s in ens.scenes:
        pos, vel = s.pos.copy(), s.vel.copy()
        pos[:, :3] += rng.uniform(-0.05 * s.info["h"], 0.05 * s.info["h"], (s.n, 3)).astype(np.float32)
        vel[:, :3] = rng.normal(0.0, 0.05, (s.n, 3))
        moved.append(scenes.Scene(s.name, pos, vel, s.fluid, s.common, s.kernels, s.key_mode, s.steps, s.seed, s.info))
    return dict(kind=kind, ens=scenes.Ensemble(moved, ens.seed, ens.bodies), steps=case["steps"])


_ORIGIN = (-0.4, -0.1, -0.4)


def _mesh(case, seed):
    v, t = mesh.torus_mesh(0.3, 0.1, case["nu"], case["nv"])
    rng = np.random.default_rng(seed)
    return (v + rng.normal(0.0, 5e-4, v.shape)).astype(np.float32), t.astype(np.uint32)


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------

def run(st):
    L = lib.load()
    kind = st["kind"]
    if kind == "steps":
        sim, out = st["kept"]["sim"], st["kept"]["out"]
        L.fg_set_stream(sim.stream())
        L.fg_copy_bytes(sim.buffers.position, st["pos"].data_ptr(), st["bytes"])
        L.fg_copy_bytes(sim.buffers.velocity, st["vel"].data_ptr(), st["bytes"])
        L.fg_set_stream(None)
        sim.step(st["steps"])
        return out
    if kind == "launchers":
        sc, g, n = st["sc"], st["g"], st["sc"]["n"]
        st["pos_out"].copy_(st["pos"])
        _sort_into_cells(sc, g, st["pos"], st["vel"])
        L.gCalcMassDensity(g.spos.data_ptr(), g.rho.data_ptr(), g.keys.data_ptr(), g.start.data_ptr(), g.end.data_ptr(),
                           n, sc["k"], sc["rho0"], sc["mass"])
        L.gSPHCalculateForces(g.spos.data_ptr(), g.svel.data_ptr(), None, g.rho.data_ptr(), g.start.data_ptr(),
                              g.end.data_ptr(), st["vel_out"].data_ptr(), g.ids.data_ptr(), n, sc["mass"], sc["mu"])
        L.gSPHIntegrate(st["pos_out"].data_ptr(), st["vel_out"].data_ptr(), None, n, g.rho.data_ptr(),
                        g.start.data_ptr(), g.end.data_ptr())
        lib.check(0, "launchers")
        return dict(pos=st["pos_out"], vel=st["vel_out"], rho_p=g.rho, ids=g.ids, keys=g.keys)
    if kind == "layers":
        sc, g, n = st["sc"], st["g"], st["sc"]["n"]
        lib.check(L.fg_sph_density_nbr(g.spos.data_ptr(), g.svel.data_ptr(), g.rho.data_ptr(), g.start.data_ptr(),
                                       g.end.data_ptr(), st["nbr"].data_ptr(), n, sc["k"], sc["rho0"], sc["mass"]))
        lib.check(L.fg_sph_forces_integrate_nbr(g.spos.data_ptr(), g.svel.data_ptr(), g.rho.data_ptr(),
                                                g.start.data_ptr(), g.end.data_ptr(), st["nbr"].data_ptr(),
                                                st["vel_out"].data_ptr(), st["pos_out"].data_ptr(), g.ids.data_ptr(),
                                                n, sc["mass"], sc["mu"]))
        return dict(pos=st["pos_out"], vel=st["vel_out"], rho_p=g.rho)
    if kind == "coupled":
        return _run_coupled(L, st)
    if kind == "sort":
        st["k"].copy_(st["keys"])
        st["v"].copy_(st["vals"])
        lib.check(L.fg_sort_pairs_ws(st["k"].data_ptr(), st["v"].data_ptr(), st["n"], st["bits"], st["ws"].data_ptr(),
                                     st["ws_bytes"], 0))
        return [st["k"], st["v"]]
    if kind == "mesh":
        lib.check(L.fg_mesh_winding_lattice(st["v"].data_ptr(), len(st["v"]), st["t"].data_ptr(), len(st["t"]),
                                            abi.f3(*_ORIGIN), st["spacing"], *st["dims"], st["out"].data_ptr()))
        return st["out"]
    sim = lib.BatchSimulator(st["ens"])
    try:
        for k, b in enumerate(st["ens"].bodies or []):
            if b is not None:
                sim.add_bodies(k, b)
        sim.step(st["steps"])
        pos, vel = sim.state()
        rho_p, _ = sim.density()
        out = dict(pos=pos, vel=vel, rho_p=rho_p)
        if st["ens"].bodies:
            out["bodies"] = sim.body_state()["pos"]
        return out
    finally:
        sim.close()


def _run_coupled(L, st):
    sc, g, b, n = st["sc"], st["g"], st["b"], st["sc"]["n"]
    torus, post = st["torus"], st["post"]
    torus.build(b, st["cm"], st["orient"])
    _sort_into_cells(sc, g, st["pos"], st["vel"])
    lib.check(L.fg_sph_density_nbr(g.spos.data_ptr(), g.svel.data_ptr(), g.rho.data_ptr(), g.start.data_ptr(),
                                   g.end.data_ptr(), st["nbr"].data_ptr(), n, sc["k"], sc["rho0"], sc["mass"]))
    dyn = _body_grid(b, torus.start, torus.end, torus.sorted, torus.bounds, st["bvel"], torus.m)
    static = _body_grid(b, post.start, post.end, post.sorted, post.bounds, None, post.m)
    cell = abi.f3(sc["cell"], sc["cell"], sc["cell"])
    lib.check(L.fg_body_forces_from_fluid(torus.world.data_ptr(), st["bvel"].data_ptr(), st["cm"].data_ptr(),
                                          st["pf"].data_ptr(), st["pt"].data_ptr(), torus.m, 1, b["radius"],
                                          g.spos.data_ptr(), g.svel.data_ptr(), g.start.data_ptr(), g.end.data_ptr(),
                                          n, b["fluid_radius"], cell, sc["buckets"], abi.i3(1, 1, 1), b["spring"],
                                          b["damping"]))
    lib.check(L.fg_body_forces_from_bodies(torus.world.data_ptr(), st["bvel"].data_ptr(), st["cm"].data_ptr(),
                                           st["pf"].data_ptr(), st["pt"].data_ptr(), torus.m, 1, b["radius"], None,
                                           None, C.byref(static), 1))
    lib.check(L.fg_sph_forces_coupled(g.spos.data_ptr(), g.svel.data_ptr(), g.rho.data_ptr(), g.start.data_ptr(),
                                      g.end.data_ptr(), st["nbr"].data_ptr(), st["vel_out"].data_ptr(),
                                      st["pos_out"].data_ptr(), g.ids.data_ptr(), n, sc["mass"], sc["mu"],
                                      C.byref(dyn), C.byref(static)))
    lib.check(L.fg_body_reduce_f64(st["pf"].data_ptr(), st["pt"].data_ptr(), st["offsets"].data_ptr(), 1,
                                   st["sums"][0].data_ptr(), st["sums"][1].data_ptr(), None, None))
    return dict(pos=st["pos_out"], vel=st["vel_out"], rho_p=g.rho, ids=g.ids, force=st["pf"], torque=st["pt"],
                sums=st["sums"])


# ---------------------------------------------------------------------------
# exact: the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

_MOST_EXACT = 9_000_000  # particles


class _Cells:
    """Points sorted by cell key, and the ranges of the 27 cells around others."""

    def __init__(self, mode, pos32, cell, vmin, dims, buckets):
        self.mode, self.dims, self.buckets = mode, dims, buckets
        self.cell = torch.tensor(cell, dtype=torch.float32, device=DEV)
        self.vmin = torch.tensor(vmin, dtype=torch.float32, device=DEV)
        keys = self.key(pos32, (0, 0, 0))
        self.order = torch.argsort(keys, stable=True)
        self.sorted = keys[self.order]

    def key(self, p, off):
        if self.mode == "xor":
            q = p + self.cell * torch.tensor(off, dtype=torch.float32, device=DEV)
            c = ((q + 5000.0) / self.cell).trunc().long()
            x = (c[:, 0] * 73856093) & 0xFFFFFFFF
            x = x ^ ((c[:, 1] * 19349663) & 0xFFFFFFFF)
            return (x ^ ((c[:, 2] * 83492791) & 0xFFFFFFFF)) % self.buckets
        top = torch.tensor(self.dims, device=DEV) - 1
        c = torch.minimum(((p - self.vmin) / self.cell).floor().long().clamp(min=0), top)
        c = c + torch.tensor(off, device=DEV)
        k = c[:, 0] + self.dims[0] * (c[:, 1] + self.dims[1] * c[:, 2])
        return torch.where(((c >= 0) & (c <= top)).all(1), k, -1)

    def pairs(self, p32):
        """Yields (i, j): the points p32[i] and the sorted points j around them."""
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    k = self.key(p32, (dx, dy, dz))
                    lo = torch.searchsorted(self.sorted, k)
                    count = torch.searchsorted(self.sorted, k, right=True) - lo
                    i = torch.nonzero(count).squeeze(1)
                    m = 0
                    while len(i):
                        yield i, lo[i] + m
                        m += 1
                        i = i[count[i] > m]


def _walls(sc, p, v):
    """Penalty walls of the box and the friction of the fixed box -11..11, -40..200."""
    s, f = sc["s"], torch.zeros_like(p)
    reach, eps = float(F(0.003043174)), float(F(0.00001))
    for axis in range(3):
        for sign in (1.0, -1.0):
            wall = sc["vmin"][axis] if sign > 0 else sc["vmax"][axis]
            d = reach - sign * (p[:, axis] - float(F(wall))) * s
            f[:, axis] += torch.where(d > eps, sign * (20000.0 * d - 256.0 * sign * v[:, axis]), 0.0)
            wall = ((-11.0, -40.0, -11.0) if sign > 0 else (11.0, 200.0, 11.0))[axis]
            d = reach - sign * (p[:, axis] - wall) * s
            # The tangential part as the reference forms it: v minus v times its signed normal component.
            t = v - v * (sign * v[:, axis])[:, None]
            f += torch.where(((d > eps) & (t.sum(1) / 3.0 > 0.0))[:, None], -t, 0.0)
    return f


def _contact(b, cells, spheres, svel, p, v, p32, mind, skip=None):
    """Penalty force on the points p from the spheres of a grid."""
    f = torch.zeros_like(p)
    for i, j in cells.pairs(p32):
        rel = spheres[j] - p[i]
        l = rel.norm(dim=1)
        n = rel / l[:, None].clamp(min=1e-300)
        c = b["spring"] * l - b["damping"] * (n * (svel[j] - v[i])).sum(1)
        f.index_add_(0, i, torch.where((l < mind)[:, None], c[:, None] * n, 0.0))
    return f


def _exact_step(sc, pos, vel, extra=None):
    """One step in 64 bits: positions, velocities and (rho, p) in particle
    order, and the sorted order; extra(cells, p, v) adds an acceleration."""
    n, s, h = sc["n"], sc["s"], sc["h"]
    p32 = pos.float()
    cells = _Cells(sc["mode"], p32, [sc["cell"]] * 3, sc["vmin"], sc["dims"], sc["buckets"])
    o = cells.order
    ps, vs, p32 = pos[o], vel[o], p32[o]
    x = ps * s
    rho = torch.zeros(n, dtype=torch.float64, device=DEV)
    for i, j in cells.pairs(p32):
        d = x[i] - x[j]
        r2 = (d * d).sum(1)
        rho.index_add_(0, i, torch.where(r2 < h * h, (h * h - r2).clamp(min=0.0) ** 3, 0.0))
    rho = rho * sc["mass"] * sc["poly6"]
    pr = sc["k"] * (rho - sc["rho0"])
    rho = rho.clamp(min=1.0)
    a = torch.zeros_like(ps)
    for i, j in cells.pairs(p32):
        d = x[i] - x[j]
        l = d.norm(dim=1)
        near = (l < h) & (i != j)
        w = (h - l) / (rho[i] * rho[j])
        cp = -sc["spiky"] * (h - l) * w * (pr[i] + pr[j]) / l.clamp(min=1e-300)
        t = cp[:, None] * d + (sc["visc"] * sc["mu"] * w)[:, None] * (vs[j] - vs[i])
        a.index_add_(0, i, torch.where(near[:, None], t, 0.0))
    a = a * sc["mass"]
    a[:, 1] += sc["g"]
    if extra is not None:
        a = a + extra(ps, vs, p32)
    a = a + _walls(sc, ps, vs)
    speed = a.norm(dim=1, keepdim=True)
    a = torch.where(speed > sc["limit"], a * (sc["limit"] / speed), a)
    v1 = torch.empty_like(vel)
    p1 = torch.empty_like(pos)
    v1[o] = vs + a * sc["dt"]
    p1[o] = ps + v1[o] * (sc["dt"] / s)
    return p1, v1, torch.stack([rho, pr], 1), cells


def _with_w(p, w):
    return torch.cat([p, torch.full((len(p), 1), w, dtype=p.dtype, device=p.device)], 1)


def exact(case, seed):
    case = _full(case)
    kind = case["kind"]
    if kind in ("steps", "launchers", "layers", "coupled"):
        sc = _scene(case)
        if sc["n"] > _MOST_EXACT:
            return None
        pos, vel = _fluid(sc, case["order"], seed)
        p, v = pos[:, :3].double(), vel[:, :3].double()
        steps, extra, more = case.get("steps", 1), None, {}
        if kind == "coupled":
            extra, more = _exact_bodies(case, sc, p, v)
        for _ in range(steps):
            p, v, rho, _ = _exact_step(sc, p, v, extra)
        out = dict(pos=_with_w(p, 1.0), vel=_with_w(v, 0.0), rho_p=rho if steps == 1 else None, **more)
        if kind != "layers":
            out["ids"] = None
        if kind == "launchers":
            out["keys"] = None
        return out
    if kind == "mesh":
        return _exact_mesh(case, seed)
    return None  # whole numbers, or a run of many scenes


def _exact_bodies(case, sc, p, v):
    b = _bodies(case, sc)
    mind = b["fluid_radius"] + b["radius"] + 0.003
    bv = torch.tensor([0.1, -0.4, 0.05], device=DEV).double()

    def grid(spheres):
        s32 = torch.from_numpy(spheres[:, :3].copy()).to(DEV)
        cells = _Cells("xor", s32, [b["cell"]] * 3, (0.0, 0.0, 0.0), None, b["buckets"])
        return cells, s32[cells.order].double()

    torus = b["torus"].copy()
    torus[:, :3] = (torus[:, :3] - b["centre"]) + b["centre"]
    (tc, ts), (pc, ps) = grid(torus), grid(b["post"])

    def extra(q, u, q32):
        return (_contact(b, pc, ps, torch.zeros_like(ps), q, u, q32, mind) +
                _contact(b, tc, ts, bv.expand_as(ts), q, u, q32, mind))

    w32 = torch.from_numpy(torus[:, :3].copy()).to(DEV)
    w = w32.double()
    fluid = _Cells(sc["mode"], p.float(), [sc["cell"]] * 3, sc["vmin"], sc["dims"], sc["buckets"])
    f = _contact(b, fluid, p[fluid.order], v[fluid.order], w, bv.expand_as(w), w32, b["fluid_radius"] + b["radius"] +
                 0.0001)
    f = f + _contact(b, pc, ps, torch.zeros_like(ps), w, bv.expand_as(w), w32, 2.0 * b["radius"] + 0.001)
    t = torch.linalg.cross(w - torch.from_numpy(b["centre"]).to(DEV).double(), f)
    sums = torch.stack([_with_w(f.sum(0, keepdim=True), 0.0), _with_w(t.sum(0, keepdim=True), 0.0)])
    return extra, dict(force=_with_w(f, 0.0), torque=_with_w(t, 0.0), sums=sums)


def _exact_mesh(case, seed):
    v, t = _mesh(case, seed)
    spacing, (nx, ny, nz), _ = _mesh_size(case)
    s = float(F(spacing))
    o = [float(F(a)) for a in _ORIGIN]
    i = torch.arange(nx * ny * nz, device=DEV)
    # the lattice points are FP32 positions
    idx = torch.stack([i % nx, (i // nx) % ny, i // (nx * ny)], 1).float()
    pts = (idx * torch.tensor(s, dtype=torch.float32, device=DEV) +
           torch.tensor(o, dtype=torch.float32, device=DEV)).double()
    tri = torch.from_numpy(v.astype(np.float64)[t.astype(np.int64)]).to(DEV)
    out = torch.empty(len(pts), dtype=torch.float64, device=DEV)
    step = max(1, 40_000_000 // len(tri))
    for k in range(0, len(pts), step):
        q = pts[k:k + step, None, :]
        a, b, c = (tri[None, :, m] - q for m in range(3))
        la, lb, lc = a.norm(dim=2), b.norm(dim=2), c.norm(dim=2)
        det = (a * torch.linalg.cross(b, c)).sum(2)
        den = la * lb * lc + (a * b).sum(2) * lc + (b * c).sum(2) * la + (c * a).sum(2) * lb
        out[k:k + step] = torch.atan2(det, den).sum(1) / (2.0 * math.pi)
    return out
