"""Timed cases of the framework: what a program that uses it has it do.

A case is a plain dict; `prepare` makes its inputs from a seed, `run` is one
pass through the public entry points, `exact` computes the same outputs in
binary64 with plain torch.  Kinds:

  substeps  DFSPHSolver.advance, or step where the divergence solve is on:
            the CFL substeps of one scene, from the same state in every pass
  batch     BatchSolver.step over many independent box scenes
  rollout   a checkpointed differentiable rollout, forward and backward
  grid      CellGrid.build
  lbvh      SpatialAccel.build
  mesh      SurfaceMesher.run on one frame of particles

Fluid states are either the lattice block at rest that every scene starts
from, or (`stirred`) what a scene looks like after some motion: the block
sheared by volume-preserving maps along the tank (so particle indices no
longer follow the cells), a few percent of jitter, and a divergence-free
velocity field of a few modes.
"""
import math

import numpy as np
import torch  # before the library loads: both then use torch's HIP runtime

import water_simulation_amd as ws
from water_simulation_amd import adjoint, mesh, scenes

DEV = "cuda"
RHO0 = 1000.0
V_MAX = 5.0      # the advection's speed limit, m/s
CLAMP = 1e-3     # its distance to the domain's faces, m
DAMPING = 0.5
ETA = 1e-3
# Stirred blocks: lattice spacing over the particle diameter that leaves the
# solve with the mean density error it meets in long runs: 2 to 4 iterations
# with kappa/rho, about 25 kg/m^3 at the cap with the reference's form.
PACK = {0: 0.985, 1: 0.998}


# ---- the cases --------------------------------------------------------------

def _sub(name, dims, radius, tank, stirred, substeps, fast, form, divergence=False, tension=0.0,
         origin=None, cap=100):
    nx, ny, nz = dims
    c = dict(kind="substeps", nx=nx, ny=ny, nz=nz, radius=radius, tx=tank[0], ty=tank[1],
             tz=tank[2], stirred=stirred, substeps=substeps, fast=fast, form=form,
             divergence=divergence, tension=tension, cap=cap)
    c["ox"], c["oy"], c["oz"] = origin or (0.0, 0.0, 0.0)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest scene that ships with the tests (single_drop): 180
        # particles in mid-air of the unit box, the simulator's own settings
        # (reference pressure form, bit-exact arithmetic).  Latency only.
        _sub("drop_180", (6, 5, 6), 0.01, (1.0, 1.0, 1.0), False, 8, False, 0,
             origin=(0.45, 0.3, 0.45)),
        # The test scene dam_break some frames in, as the simulator runs it:
        # with the reference's pressure form a substep goes to the iteration
        # cap, so the pressure sweeps are nearly all of it.
        _sub("dam_5k_capped", (11, 28, 17), 0.012, (1.0, 1.0, 1.0), True, 2, False, 0),
        # dam_break_hires with the two opt-in physics options: divergence
        # solve (step by step through the store) and surface tension.
        _sub("dam_17k_options", (16, 41, 26), 0.008, (1.0, 1.0, 1.0), True, 2, False, 1,
             divergence=True, tension=0.0728),
        # The mid dam break in its collapse, tolerance mode.
        _sub("mid_128k_fast", (40, 80, 40), 0.005, (1.6, 0.9, 0.8), True, 4, True, 1),
        # The large dam break from its lattice, bit-exact arithmetic: the
        # first frame of a long run.
        _sub("large_1m_exact", (100, 100, 100), 0.0025, (2.0, 1.0, 1.0), False, 4, False, 1),
        # The large dam break in its collapse, tolerance mode: the production
        # run (an odd particle count, fluid across the whole tank width).
        _sub("large_1m_fast", (105, 51, 187), 0.0025, (2.0, 1.0, 1.0), True, 3, True, 1),
        # 64 uneven box scenes stepped together (parameter sweeps, datasets).
        dict(name="batch_64", kind="batch", scenes=64, n_min=2000, n_max=60000, fast=True),
        # The inverse problem: a 32^3 block, a segment of its rollout and the
        # gradients with respect to its initial state and viscosity.
        dict(name="rollout_32k", kind="rollout", side=32, substeps=6, every=3),
        # Neighbour grid alone, a mid-sized odd point count.
        dict(name="grid_100k", kind="grid", n=100003, radius=0.005, tx=1.6, ty=0.9, tz=0.8),
        # Bounding volume hierarchy over a large frame.
        dict(name="lbvh_1m", kind="lbvh", n=1000000, radius=0.0025, tx=2.0, ty=1.0, tz=1.0),
        # Surface meshes of a small and a large frame, the tool's defaults.
        dict(name="mesh_17k", kind="mesh", nx=16, ny=41, nz=26, radius=0.008, tx=1.0, ty=1.0,
             tz=1.0, k=15, sigma=2.5),
        dict(name="mesh_1m", kind="mesh", nx=105, ny=51, nz=187, radius=0.0025, tx=2.0, ty=1.0,
             tz=1.0, k=15, sigma=2.5),
    ]


# tank and radius of the scenes of the configurations and tests
_TANKS = [(0.0025, (2.0, 1.0, 1.0)), (0.005, (1.6, 0.9, 0.8)), (0.008, (1.0, 1.0, 1.0)),
          (0.012, (1.0, 1.0, 1.0))]


def _block(rng, radius, tank, lo, hi):
    """Lattice dims of a block of about n particles, log-uniform in [lo, hi],
    that fits the tank with room to move along x."""
    s = 2.0 * radius
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    fit = [int((t - 8.0 * s) / s) for t in tank]
    fit[0] = int(0.6 * fit[0])
    nz = min(fit[2], max(3, int(n ** (1 / 3) * rng.uniform(0.6, 1.8))))
    ny = min(fit[1], max(3, int((n / nz) ** 0.5 * rng.uniform(0.6, 1.6))))
    nx = min(fit[0], max(3, int(n / (nz * ny))))
    return nx, ny, nz


def draw(rng):
    kind = rng.choice(["substeps"] * 6 + ["batch", "rollout", "grid", "lbvh", "mesh", "mesh"])
    radius, tank = rng.choice(_TANKS)
    top = {0.0025: 1000000, 0.005: 200000, 0.008: 60000, 0.012: 20000}[radius]
    if kind in ("grid", "lbvh"):
        n = int(math.exp(rng.uniform(math.log(100), math.log(1000000)))) | 1
        return dict(kind=kind, n=n, radius=radius, tx=tank[0], ty=tank[1], tz=tank[2])
    if kind == "batch":
        lo = rng.randrange(200, 4000)
        return dict(kind="batch", scenes=rng.randrange(3, 65), n_min=lo,
                    n_max=lo * rng.randrange(2, 12), fast=rng.random() < 0.5)
    if kind == "rollout":
        return dict(kind="rollout", side=rng.randrange(7, 33), substeps=rng.randrange(2, 7),
                    every=rng.randrange(1, 5))
    if kind == "mesh":
        nx, ny, nz = _block(rng, radius, tank, 500, 0.5 * top)
        return dict(kind="mesh", nx=nx, ny=ny, nz=nz, radius=radius, tx=tank[0], ty=tank[1],
                    tz=tank[2], k=rng.choice([8, 10, 15, 15, 15, 20]),
                    sigma=rng.choice([2.25, 2.5, 2.5, 2.5, 3.0]))
    form = 0 if top <= 60000 and rng.random() < 0.4 else 1
    dims = _block(rng, radius, tank, 60, top)
    return _sub(None, dims, radius, tank, rng.random() < 0.8, rng.randrange(1, 5),
                rng.random() < 0.5, form, divergence=form == 1 and rng.random() < 0.2,
                tension=0.0728 if rng.random() < 0.2 else 0.0, cap=rng.choice([20, 50, 100]))


# ---- inputs -----------------------------------------------------------------

def _lattice(case):
    """Lattice indices of the block, x-major, and its spacing."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    s = 2.0 * case["radius"]
    i = torch.arange(nx * ny * nz, device=DEV)
    ijk = torch.stack([i // (ny * nz), (i // nz) % ny, i % nz], 1).double()
    return ijk, s


def fluid_state(case, seed):
    """(x, v), binary32, n x 3, on the GPU."""
    ijk, s = _lattice(case)
    g = torch.Generator().manual_seed(seed * 7919 + 17)
    rnd = lambda *k: torch.rand(*k, generator=g, dtype=torch.float64)  # noqa: E731
    noise = torch.Generator(device=DEV).manual_seed(seed * 104729 + 5)
    if not case.get("stirred", True):
        org = [case["ox"], case["oy"], case["oz"]]
        first = torch.tensor([o if o > 0.0 else 3.0 * s for o in org], dtype=torch.float32,
                             device=DEV)
        x = first + np.float32(s) * ijk.float()
        v = 0.02 * torch.randn(x.shape, generator=noise, device=DEV, dtype=torch.float64)
        v[:, 1] -= 0.3
        return x, v.float()
    s = PACK[case.get("form", 1)] * s
    n = [case["nx"], case["ny"], case["nz"]]
    tank = [case["tx"], case["ty"], case["tz"]]
    wall = 3.0 * 2.0 * case["radius"]  # the first slot clear of the wall layers
    span = [(k - 1) * s for k in n]
    room = [max(0.0, t - 2.0 * wall - d) for t, d in zip(tank, span)]
    u = ijk * s
    # x by functions of (y, z), then z by functions of (x, y): each preserves volume
    ax = 0.5 * room[0] * 0.6
    ph = 2.0 * math.pi * rnd(4)
    wz = 2.0 * math.pi / max(span[2], 4.0 * s)
    wy = 2.0 * math.pi / max(span[1], 4.0 * s)
    lim = 0.5 / max(wz, wy)  # shear of at most one half
    ax = min(ax, lim)
    x0 = u[:, 0] + ax * (2.0 + torch.sin(wz * u[:, 2] + ph[0].item()) +
                         torch.sin(wy * u[:, 1] + ph[1].item()))
    wx = 2.0 * math.pi / max(span[0], 4.0 * s)
    az = min(0.5 * room[2], 0.5 / wx)
    z0 = u[:, 2] + 0.5 * room[2] + az * torch.sin(wx * x0 + ph[2].item())
    x = torch.stack([x0, u[:, 1], z0], 1) + wall
    x += 0.02 * s * (torch.rand(x.shape, generator=noise, device=DEV, dtype=torch.float64) - 0.5)
    for a in range(3):
        x[:, a].clamp_(wall, tank[a] - wall)
    # curls of stream functions that vanish on the block's faces
    lo = x.min(0).values
    ext = (x.max(0).values - lo).clamp_min(s)
    w = (x - lo) / ext
    v = torch.zeros_like(x)
    for a, b in ((0, 1), (1, 2), (2, 0)):
        for _ in range(2):
            ka, kb = int(1 + 2 * rnd(1).item()), int(1 + 2 * rnd(1).item())
            amp = (rnd(1).item() - 0.5)
            pa, pb = math.pi * ka, math.pi * kb
            sa, ca = torch.sin(pa * w[:, a]), torch.cos(pa * w[:, a])
            sb, cb = torch.sin(pb * w[:, b]), torch.cos(pb * w[:, b])
            v[:, a] += amp * sa * cb * (pb / ext[b])
            v[:, b] -= amp * ca * sb * (pa / ext[a])
    v *= 1.5 / v.norm(dim=1).max()
    v += 0.01 * torch.randn(v.shape, generator=noise, device=DEV, dtype=torch.float64)
    return x.float(), v.float()


def config(case):
    r = case["radius"]
    return dict(rest_density=RHO0, particle_radius=r, smoothing_length=2.0 * r, viscosity=0.01,
                damping=DAMPING, surface_tension=case["tension"], max_density_iters=case["cap"],
                max_divergence_iters=case["cap"], eta_density=ETA, eta_divergence=ETA,
                domain_min=(0.0, 0.0, 0.0), domain_max=(case["tx"], case["ty"], case["tz"]),
                enable_divergence_solve=case["divergence"], pressure_form=case["form"],
                enable_surface_tension=case["tension"] > 0.0, fast_math=case["fast"])


def box_scenes(case, seed):
    """The seeded uneven mix (the same blocks in every pass), velocities from the seed."""
    mix = scenes.uneven_mix(case["scenes"], n_min=case["n_min"], n_max=case["n_max"])
    rng = np.random.default_rng(seed)
    for m in mix:
        m.velocities = rng.normal(0.0, 0.5, m.positions.shape).astype(np.float32)
    return mix


class _Memory:
    """Device memory of the library as torch.as_tensor takes it."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr,
                                             data=(ptr, False), version=2)


def _view(ptr, shape, typestr, owner):
    if not ptr or 0 in shape:
        dt = torch.int32 if typestr == "<i4" else torch.float32
        return torch.empty(shape, dtype=dt, device=DEV)
    return torch.as_tensor(_Memory(ptr, shape, typestr, owner), device=DEV)


def _store(x):
    st = ws.ParticleStore(len(x))
    st.resize(len(x))
    if isinstance(x, np.ndarray):
        st.set_positions(x)
    else:
        _view(st.positions(), x.shape, "<f4", st).copy_(x)
    return st


def _dt_max(radius):
    """The scenes' largest substep: the CFL step at the speed limit, so that a
    pass does not depend on the speed that the one before ended with."""
    return 0.4 * radius / V_MAX


def _walls(tank, radius):
    return ws.sample_aabb_boundary((0.0, 0.0, 0.0), tank, 2.0 * radius, 3)


def _points(case, seed):
    """A cloud that fills the lower half of the tank, in no order."""
    g = torch.Generator(device=DEV).manual_seed(seed * 15485863 + 3)
    t = torch.tensor([case["tx"], 0.5 * case["ty"], case["tz"]], device=DEV)
    return torch.rand((case["n"], 3), generator=g, device=DEV) * t


def _fields(store, n, divergence=False):
    out = {"x": _view(store.positions(), (n, 3), "<f4", store),
           "v": _view(store.velocities(), (n, 3), "<f4", store)}
    names = ["density", "alpha", "kappa", "density_adv"] + (["kappa_v"] if divergence else [])
    for k in names:
        h = store.find_attribute("dfsph_" + k)
        out[k] = _view(store.attribute_data(h), (n,), "<f4", store)
    return out


def prepare(case, seed):
    torch.zeros(1, device=DEV)
    kind = case["kind"]
    s = {"case": case}
    if kind == "substeps":
        s["x0"], s["v0"] = fluid_state(case, seed)
        n = len(s["x0"])
        s["fluid"] = _store(s["x0"])
        s["walls"] = _store(_walls((case["tx"], case["ty"], case["tz"]), case["radius"]))
        s["solver"] = ws.DFSPHSolver(s["fluid"], s["walls"], ws.DFSPHConfig(**config(case)))
        s["stepper"] = ws.TimeStepper(ws.TimeStepperConfig(dt_max=_dt_max(case["radius"])))
        s["out"] = _fields(s["fluid"], n, case["divergence"])
    elif kind == "batch":
        mix = box_scenes(case, seed)
        s["x0"] = torch.from_numpy(np.concatenate([m.positions for m in mix])).to(DEV)
        s["v0"] = torch.from_numpy(np.concatenate([m.velocities for m in mix])).to(DEV)
        s["fluid"] = _store(s["x0"])
        s["walls"] = _store(_walls((scenes.BOX,) * 3, scenes.RADIUS))
        cfg = ws.DFSPHConfig(**scenes.box_config(pressure_form=1, fast_math=case["fast"]))
        s["solver"] = ws.BatchSolver(s["fluid"], s["walls"], cfg, [len(m.positions) for m in mix],
                                     [m.viscosity for m in mix])
        s["solver"].set_graphs(False)  # eager launches, the faster mode on this device
        s["dt"] = _batch_dts(mix)
        s["out"] = _fields(s["fluid"], len(s["x0"]))
    elif kind == "rollout":
        x0, v0, gx, gv = _rollout_inputs(case, seed)
        s["x0"], s["v0"] = x0.requires_grad_(), v0.requires_grad_()
        s["eps"] = torch.tensor(0.01, dtype=torch.float64, device=DEV, requires_grad=True)
        s["g"] = (gx, gv)
        s["fluid"] = _store(x0.detach())
        s["walls"] = _store(_walls((adjoint.BOX,) * 3, adjoint.RADIUS))
        cfg = ws.DFSPHConfig(**adjoint.inverse_config())
        s["solver"] = ws.DFSPHSolver(s["fluid"], s["walls"], cfg)
        s["rollout"] = adjoint.Rollout(s["solver"], checkpoint_every=case["every"])
        s["fn"] = adjoint.rollout_function()
        s["dts"] = np.full(case["substeps"], adjoint.DT, np.float32)
    elif kind == "grid":
        s["x"] = _points(case, seed)
        l = 2.0 * case["radius"]
        dims = [int(math.ceil(t / l)) + 2 for t in (case["tx"], case["ty"], case["tz"])]
        s["grid"] = ws.CellGrid((-l, -l, -l), dims, l)
        s["grid"].reserve(case["n"])
    elif kind == "lbvh":
        s["x"] = _points(case, seed)
        s["accel"] = ws.SpatialAccel()
        s["lo"], s["hi"] = (0.0, 0.0, 0.0), (case["tx"], case["ty"], case["tz"])
    else:
        s["x"] = fluid_state(case, seed)[0]
        s["mesher"] = mesh.SurfaceMesher()
        # the buffers that a renderer or a writer keeps for a frame's mesh
        cap = int(3 * _mesh_vertices(case)) + 8 * len(s["x"]) + 4096
        s["vertices"] = torch.zeros((cap, 3), device=DEV)
        s["triangles"] = torch.zeros((2 * cap, 3), dtype=torch.int32, device=DEV)
    return s


def _batch_dts(mix):
    ts = ws.TimeStepper()
    return np.array([ts.next_dt(max(scenes.initial_max_speed(m.velocities), 0.5), scenes.RADIUS,
                                1.0) for m in mix], np.float32)


def _rollout_inputs(case, seed):
    """A block a little off its lattice, a smooth velocity, and the gradients
    of a loss that varies smoothly over the block."""
    x = adjoint.block_positions(case["side"])
    rng = np.random.default_rng(seed)
    x = (x + rng.uniform(-1e-4, 1e-4, x.shape)).astype(np.float32)
    f = [adjoint.smooth_velocity(x, 3 * seed + k, amplitude=a)
         for k, a in ((0, 0.5), (1, 1.0), (2, 0.01))]
    return [torch.from_numpy(a).to(DEV) for a in [x] + f]


# ---- one pass ---------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("substeps", "batch"):
        s["out"]["x"].copy_(s["x0"])  # the state that the pass starts from
        s["out"]["v"].copy_(s["v0"])
    if kind == "substeps":
        dts = s["solver"].advance(1e9, case["substeps"], s["stepper"], v_floor=0.5)
        return dict(s["out"], dts=dts)
    if kind == "batch":
        s["solver"].step(s["dt"])
        return s["out"]
    if kind == "rollout":
        xT, vT = s["fn"].apply(s["x0"], s["v0"], s["eps"], s["rollout"], s["dts"])
        gx0, gv0, ge = torch.autograd.grad((xT, vT), (s["x0"], s["v0"], s["eps"]), s["g"])
        return {"x": xT.detach(), "v": vT.detach(), "gx0": gx0, "gv0": gv0, "ge": ge}
    if kind == "grid":
        g = s["grid"]
        g.build(s["x"].data_ptr(), case["n"])
        return {"keys": _view(g.sorted_keys(), (case["n"],), "<i4", g),
                "indices": _view(g.sorted_indices(), (case["n"],), "<i4", g),
                "cell_start": _view(g.cell_start(), (g.total_cells() + 1,), "<i4", g)}
    L = ws._ffi.lib()
    if kind == "lbvh":
        a, n = s["accel"], case["n"]
        a.build(s["x"].data_ptr(), n, s["lo"], s["hi"])
        return {"indices": _view(L.wsim_accel_sorted_indices(a._h), (n,), "<i4", a),
                "codes": _view(L.wsim_accel_morton_codes(a._h), (n,), "<i4", a),
                "left": _view(L.wsim_accel_internal_left(a._h), (n - 1,), "<i4", a),
                "right": _view(L.wsim_accel_internal_right(a._h), (n - 1,), "<i4", a),
                "parent": _view(L.wsim_accel_internal_parent(a._h), (2 * n - 1,), "<i4", a),
                "boxes": _view(L.wsim_accel_node_aabbs(a._h), (2 * n - 1, 2, 3), "<f4", a)}
    m = s["mesher"]
    info = m.run((s["x"].data_ptr(), len(s["x"])), radius=case["radius"],
                 smooth_sigma=case["sigma"], k_neighbors=case["k"])
    ptr = ws._ffi.C.c_void_p()
    for name, fn, typestr in (("vertices", L.wsim_mesher_vertices, "<f4"),
                              ("triangles", L.wsim_mesher_triangles, "<i4")):
        ws._ffi.check(fn(m._h, ws._ffi.C.byref(ptr)))
        k = info["n_" + name]
        s[name][:k].copy_(_view(ptr.value, (k, 3), typestr, m))
    return {"vertices": s["vertices"], "triangles": s["triangles"],
            "counts": np.array([info["n_vertices"], info["n_triangles"], *info["dims"]]),
            "max_density": float(info["max_density"]), "lo": info["lo"],
            "spacing": info["spacing"]}


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    """Bytes: every input of a pass read once and every output written once.
    Operations: the pair terms of about 27 neighbours per particle (a density
    and gradient term is about 40 operations, a term of XSPH or of a sweep of
    a solve about 20), two sweeps for each iteration that a solve cannot skip."""
    kind = case["kind"]
    if kind == "substeps":
        n = case["nx"] * case["ny"] * case["nz"]
        k = case["substeps"]
        iters = case["cap"] if case["form"] == 0 and case["stirred"] else 2
        sweeps = 2 * iters + (2 if case["divergence"] else 0)
        # x, v in; x, v and the attributes out; the substeps between hold x, v
        return {"bytes": float(n * (24 + 24 * 2 * (k - 1) + 24 + 16)),
                "flops": float(n * k * 27 * (60 + 20 * sweeps))}
    if kind == "batch":
        mean = (case["n_max"] - case["n_min"]) / math.log(case["n_max"] / case["n_min"])
        n = case["scenes"] * mean
        return {"bytes": n * 64.0, "flops": n * 27.0 * (60 + 20 * 4)}
    if kind == "rollout":
        n, k = case["side"] ** 3, case["substeps"]
        return {"bytes": float(n * (24 + 24 + 24 + 24 + 48 * (k - 1))),
                "flops": float(n * k * 27 * (60 + 20 * 4) * 4)}
    if kind == "grid":
        l = 2.0 * case["radius"]
        cells = 1
        for t in (case["tx"], case["ty"], case["tz"]):
            cells *= int(math.ceil(t / l)) + 2
        return {"bytes": float(case["n"] * 20 + 4 * cells), "flops": 0.0}
    if kind == "lbvh":
        return {"bytes": float(case["n"] * (12 + 8 + 8 + 8 + 48)), "flops": 0.0}
    # the grid written once, two smoothing passes of k neighbours, three blur passes
    n = case["nx"] * case["ny"] * case["nz"]
    voxels = 1.0
    for k in (case["nx"], case["ny"], case["nz"]):
        voxels *= 4.0 * k + 16.0
    taps = 2 * int(4.0 * case["sigma"] + 0.5) + 1
    return {"bytes": 4.0 * voxels + 12.0 * n + 36.0 * _mesh_vertices(case),
            "flops": 3.0 * taps * voxels + 2.0 * n * case["k"] * 10}


def _mesh_vertices(case):
    """About one vertex for each voxel face (half a radius wide) of the block's surface."""
    a, b, c = (4.0 * (case[k] + 2) for k in ("nx", "ny", "nz"))
    return 2.0 * (a * b + b * c + c * a)


# ---- the same outputs in binary64 -------------------------------------------

class _Cells:
    """Uniform grid whose cell of a point is that of its binary32 rounding, as
    the path defines it; candidate pairs are those of the 27-cell stencil."""

    def __init__(self, lo, hi, l):
        f = np.float32
        self.l = float(f(l))
        self.inv = float(f(1.0) / f(l))
        self.lo = [float(f(a) - f(l)) for a in lo]
        self.d = [int(np.ceil((f(b) - f(a)) / f(l))) + 2 for a, b in zip(lo, hi)]

    def coords(self, x):
        o = torch.tensor(self.lo, dtype=torch.float32, device=x.device)
        c = torch.floor((x.detach().float() - o) * np.float32(self.inv))
        top = torch.tensor(self.d, dtype=torch.float32, device=x.device) + 1.0
        c = torch.where(c >= -2.0, c, torch.full_like(c, -2.0))  # NaN and far below
        return torch.minimum(c, top).long()

    def keys(self, c):
        d = self.d
        ok = (c >= 0).all(1) & (c[:, 0] < d[0]) & (c[:, 1] < d[1]) & (c[:, 2] < d[2])
        k = (c[:, 0] * d[1] + c[:, 1]) * d[2] + c[:, 2]
        return torch.where(ok, k, torch.full_like(k, d[0] * d[1] * d[2]))


def _pairs(cells, x, y, reach):
    """(i, j) with j in the 27-cell stencil of i's home cell and |x_i - y_j| < reach."""
    d = cells.d
    cx = cells.coords(x)
    key, order = torch.sort(cells.keys(cells.coords(y)), stable=True)
    out_i, out_j = [], []
    xd, yd = x.detach(), y.detach()
    lo, hi = (cx[:, 2] - 1).clamp_min(0), (cx[:, 2] + 1).clamp_max(d[2] - 1)
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            a, b = cx[:, 0] + dx, cx[:, 1] + dy
            ok = (a >= 0) & (a < d[0]) & (b >= 0) & (b < d[1]) & (lo <= hi)
            row = (a * d[1] + b) * d[2]
            s = torch.searchsorted(key, row + lo)
            e = torch.searchsorted(key, row + hi, right=True)
            cnt = torch.where(ok, e - s, torch.zeros_like(s))
            i = torch.repeat_interleave(torch.arange(len(x), device=x.device), cnt)
            if not len(i):
                continue
            first = torch.cumsum(cnt, 0) - cnt
            j = order[s[i] + torch.arange(len(i), device=x.device) - first[i]]
            near = ((xd[i] - yd[j]) ** 2).sum(1) < reach * reach
            out_i.append(i[near])
            out_j.append(j[near])
    if not out_i:
        e = torch.empty(0, dtype=torch.long, device=x.device)
        return e, e
    return torch.cat(out_i), torch.cat(out_j)


class _Dfsph:
    """One scene of the substep in binary64, differentiable, on pair lists."""

    def __init__(self, cfg, walls):
        f32 = lambda v: float(np.float32(v))  # noqa: E731
        self.cfg = cfg
        self.l = f32(np.float32(cfg["smoothing_length"]))
        r = f32(cfg["particle_radius"])
        self.mass = RHO0 * (2.0 * r) ** 3
        self.radius = r
        self.cells = _Cells(cfg["domain_min"], cfg["domain_max"], cfg["smoothing_length"])
        self.sigma = 1.0 / (math.pi * self.l ** 3)
        self.xb = torch.from_numpy(walls).to(DEV).double()
        i, j = _pairs(self.cells, self.xb, self.xb, 2.0 * self.l)
        w, _ = self.kernel((self.xb[i] - self.xb[j]).norm(dim=1))
        sw = torch.zeros(len(self.xb), dtype=torch.float64, device=DEV).index_add_(0, i, w)
        self.mb = RHO0 / sw.clamp_min(1e-9)

    def kernel(self, dist):
        """W and the factor c of grad W = r c."""
        q = dist / self.l
        t = (2.0 - q).clamp_min(0.0)
        w = torch.where(q < 1.0, 1.0 - 1.5 * q * q + 0.75 * q ** 3, 0.25 * t ** 3)
        safe = torch.where(dist > 1e-12, dist, torch.ones_like(dist))
        c = torch.where(q < 1.0, -3.0 * q + 2.25 * q * q, -0.75 * t * t) / (self.l * safe)
        return self.sigma * w, self.sigma * torch.where(dist > 1e-12, c, torch.zeros_like(c))

    def geometry(self, x):
        n = len(x)
        acc = lambda i, v: torch.zeros((n,) + v.shape[1:], dtype=torch.float64,  # noqa: E731
                                       device=x.device).index_add(0, i, v)
        i, j = _pairs(self.cells, x, x, 2.0 * self.l)
        other = i != j
        i, j = i[other], j[other]
        rij = x[i] - x[j]
        w, c = self.kernel((rij ** 2).sum(1).clamp_min(1e-300).sqrt())
        grad = rij * c[:, None]
        ib, jb = _pairs(self.cells, x, self.xb, 2.0 * self.l)
        rb = x[ib] - self.xb[jb]
        wb, cb = self.kernel((rb ** 2).sum(1).clamp_min(1e-300).sqrt())
        mgb = (self.mb[jb] * cb)[:, None] * rb
        rho = self.mass * (acc(i, w) + self.sigma) + acc(ib, self.mb[jb] * wb)
        G = self.mass * acc(i, grad) + acc(ib, mgb)
        Q = self.mass ** 2 * acc(i, (grad ** 2).sum(1)) + acc(ib, (mgb ** 2).sum(1))
        den = (G ** 2).sum(1) + Q
        alpha = torch.where(den > 1e-9, rho / den.clamp_min(1e-9), torch.zeros_like(den))
        return dict(i=i, j=j, w=w, grad=grad, r=rij, ib=ib, Gb=acc(ib, mgb), rho=rho, alpha=alpha,
                    acc=acc)

    def change(self, g, v):
        """Density rate of the velocities v."""
        d = ((v[g["i"]] - v[g["j"]]) * g["grad"]).sum(1)
        return self.mass * g["acc"](g["i"], d) + (v * g["Gb"]).sum(1)

    def solve(self, g, v, dt, cap, divergence, form):
        power = 1 if form else 2
        kap = out = torch.zeros_like(g["rho"])
        for it in range(cap):
            rd = self.change(g, v)
            out = rd if divergence else g["rho"] + dt * rd
            err = out.clamp_min(0.0) if divergence else (out - RHO0).clamp_min(0.0)
            kap = err * g["alpha"] / (dt if divergence else dt * dt)
            kh = kap / g["rho"] ** power
            t = (self.mass * (kh[g["i"]] + kh[g["j"]]))[:, None] * g["grad"]
            v = v - dt * (g["acc"](g["i"], t) + (kh + kap / RHO0 ** power)[:, None] * g["Gb"])
            if (it >= 1 or divergence) and err.detach().mean().item() < ETA * RHO0:
                break
        return v, kap, out

    def substep(self, x, v, dt, eps):
        cfg = self.cfg
        form = cfg["pressure_form"]
        g = self.geometry(x)
        i, j = g["i"], g["j"]
        grav = torch.tensor([0.0, -9.81, 0.0], dtype=torch.float64, device=x.device)
        v = v * math.exp(-cfg["damping"] * dt) + dt * grav
        k = self.mass * g["w"] / (0.5 * (g["rho"][i] + g["rho"][j]))
        v = v + eps * g["acc"](i, k[:, None] * (v[j] - v[i]))
        if cfg.get("enable_surface_tension"):
            v = v + dt * self.tension(g, cfg["surface_tension"])
        v, kap, adv = self.solve(g, v, dt, cfg["max_density_iters"], False, form)
        speed = (v.detach() ** 2).sum(1).clamp_min(1e-300).sqrt()
        fast = speed > V_MAX
        if bool(fast.any()):
            live = (v ** 2).sum(1).clamp_min(1e-300).sqrt()
            v = torch.where(fast[:, None], v * (V_MAX / live)[:, None], v)
        x = x + dt * v
        lo = torch.tensor(cfg["domain_min"], dtype=torch.float64, device=x.device) + CLAMP
        hi = torch.tensor(cfg["domain_max"], dtype=torch.float64, device=x.device) - CLAMP
        out = ((x < lo) & (v < 0)) | ((x > hi) & (v > 0))
        x = torch.minimum(torch.maximum(x, lo), hi)
        v = torch.where(out, torch.zeros_like(v), v)
        f = dict(density=g["rho"], alpha=g["alpha"], kappa=kap, density_adv=adv)
        if cfg.get("enable_divergence_solve"):
            g = self.geometry(x)
            v, kv, rd = self.solve(g, v, dt, cfg["max_divergence_iters"], True, form)
            f.update(density=g["rho"], alpha=g["alpha"], kappa_v=kv, density_adv=rd)
        return x, v, f

    def tension(self, g, gamma):
        i, j, rho = g["i"], g["j"], g["rho"]
        L = 2.0 * self.l
        nrm = L * g["acc"](i, (self.mass / rho[j])[:, None] * g["grad"])
        d = g["r"].norm(dim=1)
        t = (L - d) ** 3 * d ** 3
        C = 32.0 / (math.pi * L ** 9) * torch.where(2.0 * d > L, t, 2.0 * t - L ** 6 / 64.0)
        K = 2.0 * RHO0 / (rho[i] + rho[j])
        s = -gamma * self.mass * C / d
        a = K[:, None] * (s[:, None] * g["r"] - gamma * (nrm[i] - nrm[j]))
        return g["acc"](i, a)


def _blur64(g, sigma):
    R = int(4.0 * sigma + 0.5)
    t = torch.arange(-R, R + 1, dtype=torch.float64, device=g.device)
    w = torch.exp(-0.5 / (sigma * sigma) * t * t)
    w = w / w.sum()
    for axis in range(3):
        n = g.shape[axis]
        idx = torch.arange(-R, n + R, device=g.device) % (2 * n)
        idx = torch.where(idx >= n, 2 * n - 1 - idx, idx)
        acc = torch.zeros_like(g)
        for k in range(2 * R + 1):
            acc += w[k] * g.index_select(axis, idx[k:k + n])
        g = acc
    return g


def _smooth64(p, k):
    """Every point to the mean of its k nearest points (itself included)."""
    lo = p.min(0).values
    span = (p.max(0).values - lo).clamp_min(1e-9)
    n = len(p)
    cell = float((span.prod() / n * 2.0).pow(1.0 / 3.0))
    cell = max(cell, float(span.max()) / 1000.0)
    todo = torch.arange(n, device=p.device)
    out = torch.empty_like(p)
    while len(todo):
        d = [int(e / cell) + 1 for e in span.tolist()]
        c = ((p - lo) / cell).long()
        key = (c[:, 0] * d[1] + c[:, 1]) * d[2] + c[:, 2]
        key, order = torch.sort(key, stable=True)
        left = []
        for q in todo.split(100000):
            cq = c[q]
            best = torch.full((len(q), k), math.inf, dtype=torch.float64, device=p.device)
            who = torch.zeros((len(q), k), dtype=torch.long, device=p.device)
            zl, zh = (cq[:, 2] - 1).clamp_min(0), (cq[:, 2] + 1).clamp_max(d[2] - 1)
            for a in (-1, 0, 1):
                for b in (-1, 0, 1):
                    xa, yb = cq[:, 0] + a, cq[:, 1] + b
                    ok = (xa >= 0) & (xa < d[0]) & (yb >= 0) & (yb < d[1])
                    row = (xa * d[1] + yb) * d[2]
                    s = torch.searchsorted(key, row + zl)
                    m = torch.where(ok, torch.searchsorted(key, row + zh, right=True) - s, 0 * s)
                    width = int(m.max())
                    if not width:
                        continue
                    t = torch.arange(width, device=p.device)
                    have = t[None, :] < m[:, None]
                    j = order[torch.where(have, s[:, None] + t[None, :], 0 * s[:, None])]
                    dd = ((p[j] - p[q][:, None, :]) ** 2).sum(2)
                    dd = torch.where(have, dd, torch.full_like(dd, math.inf))
                    best, at = torch.cat([best, dd], 1).topk(k, dim=1, largest=False)
                    who = torch.cat([who, j], 1).gather(1, at)
            done = best[:, -1] < (cell * (1.0 - 1e-9)) ** 2
            out[q[done]] = p[who[done]].mean(1)
            left.append(q[~done])
        todo = torch.cat(left)
        cell *= 2.0
    return out


def _mesh64(case, seed):
    p = fluid_state(case, seed)[0].double()[:, [0, 2, 1]]
    for _ in range(2):
        p = _smooth64(p, case["k"])
    r = case["radius"]
    lo, hi = p.min(0).values - 4.0 * r, p.max(0).values + 4.0 * r
    ext = hi - lo
    res = torch.ceil(ext / (0.5 * r)).long().clamp_min(8)
    c = torch.minimum(((p - lo) / ext * res).long().clamp_min(0), res - 1)
    d = res.tolist()
    g = torch.zeros(d[0] * d[1] * d[2], dtype=torch.float64, device=DEV)
    g.index_add_(0, (c[:, 0] * d[1] + c[:, 1]) * d[2] + c[:, 2],
                 torch.ones(len(c), dtype=torch.float64, device=DEV))
    g = _blur64(g.reshape(d), case["sigma"])
    return {"vertices": None, "triangles": None, "counts": None, "max_density": float(g.max()),
            "lo": lo, "spacing": ext / res}


def exact(case, seed):
    kind = case["kind"]
    if kind == "substeps":
        cfg = config(case)
        x, v = (t.double() for t in fluid_state(case, seed))
        sim = _Dfsph(cfg, _walls((case["tx"], case["ty"], case["tz"]), case["radius"]))
        dts, vmax = [], 0.5
        with torch.no_grad():
            for _ in range(case["substeps"]):
                dt = min(_dt_max(sim.radius), 0.4 * sim.radius / max(vmax, 0.5))
                x, v, f = sim.substep(x, v, dt, cfg["viscosity"])
                vmax = float(v.norm(dim=1).max())
                dts.append(dt)
        return dict(f, x=x, v=v, dts=np.array(dts))
    if kind == "batch":
        cfg = scenes.box_config(pressure_form=1)
        sim = _Dfsph(cfg, _walls((scenes.BOX,) * 3, scenes.RADIUS))
        mix = box_scenes(case, seed)
        parts = []
        with torch.no_grad():
            for m, dt in zip(mix, _batch_dts(mix)):
                x = torch.from_numpy(m.positions).to(DEV).double()
                v = torch.from_numpy(m.velocities).to(DEV).double()
                x, v, f = sim.substep(x, v, float(dt), m.viscosity)
                parts.append(dict(f, x=x, v=v))
        return {k: torch.cat([q[k] for q in parts]) for k in parts[0]}
    if kind == "rollout":
        x0, v0, gx, gv = _rollout_inputs(case, seed)
        cfg = adjoint.inverse_config()
        sim = _Dfsph(cfg, _walls((adjoint.BOX,) * 3, adjoint.RADIUS))
        x0, v0 = x0.double().requires_grad_(), v0.double().requires_grad_()
        eps = torch.tensor(0.01, dtype=torch.float64, device=DEV, requires_grad=True)
        x, v = x0, v0
        for _ in range(case["substeps"]):
            x, v, _ = sim.substep(x, v, float(np.float32(adjoint.DT)), eps)
        gx0, gv0, ge = torch.autograd.grad((x, v), (x0, v0, eps), (gx.double(), gv.double()))
        return {"x": x.detach(), "v": v.detach(), "gx0": gx0, "gv0": gv0, "ge": ge}
    if kind == "mesh":
        return _mesh64(case, seed)
    # grids, codes and nodes are whole numbers; a node's box holds input
    # coordinates themselves (minima and maxima)
    return None
