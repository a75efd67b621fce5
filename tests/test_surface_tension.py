"""Surface tension (Akinci et al. 2013 cohesion + curvature) after XSPH.

The reference parses a surface-tension coefficient (scene/src/loader.cpp:50,
apps/sim_cli/main.cpp:132) and ships the cohesion kernel C(r, h)
(core/include/water/core/sph_kernels.cuh:44-51) but applies no force; this build applies
Akinci's force when ``enable_surface_tension`` is set (off by default, so the
default step is the reference's).

CPU: the oracle phase is pinned by the two-body closed form (every sum has one
term, n_j follows from n_i), momentum conservation on a random cluster, the
continuity of C at L/2, the off/zero-coefficient cases, and binary32 against
binary64.  GPU: the HIP step (pair lists, staged tiles, the stencil walk for
particles with coincident neighbours, graph replay, batched scenes) against
the binary32 oracle bit for bit.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

from helpers import Pair, assert_bitexact, random_box
from oracle import oracle as O

GAMMA = 0.2


def _cfg(**over):
    c = dict(rest_density=1000.0, particle_radius=0.01, smoothing_length=0.02, viscosity=0.0,
             damping=0.0, gravity=(0.0, 0.0, 0.0), domain_min=(0, 0, 0), domain_max=(1, 1, 1),
             surface_tension=GAMMA, enable_surface_tension=True)
    c.update(over)
    return c


def _f32(v):
    """A binary32 setting as the binary64 solver reads it."""
    return float(np.float32(v))


def _mass(cfg):
    return _f32(cfg["rest_density"]) * (2.0 * _f32(cfg["particle_radius"])) ** 3


def _tension_dv(x, cfg, precision=O.F64, dt=1e-3):
    """Velocity change of the surface-tension phase alone, from rest."""
    s = O.Solver(O.config(**cfg), np.asarray(x, np.float32), None, None, precision)
    dt = _f32(dt)
    s.density_alpha()
    v0 = s.get(O.FIELD_V)
    s.surface_tension(dt)
    return (s.get(O.FIELD_V) - v0) / dt, s


# --- textbook pieces, written from Akinci et al. 2013 eq. 2 and Monaghan's
# cubic spline, independent of the oracle's code; pi is the binary32 constant
# of core/include/water/core/sph_kernels.cuh:8 ------------------------------

PI = _f32(math.pi)


def _akinci_C(r, h):
    """Akinci's cohesion spline on support h."""
    k = 32.0 / (PI * h ** 9)
    if 2.0 * r > h and r <= h:
        return k * (h - r) ** 3 * r ** 3
    if 0.0 < r <= h / 2.0:
        return k * (2.0 * (h - r) ** 3 * r ** 3 - h ** 6 / 64.0)
    return 0.0


def _spline_dWdr(r, l):
    """dW/dr of the cubic spline with sigma = 1 / (pi l^3), support 2l."""
    q = r / l
    s = 1.0 / (PI * l ** 3)
    if q < 1.0:
        return s * (-3.0 * q + 2.25 * q * q) / l
    if q < 2.0:
        return -0.75 * s * (2.0 - q) ** 2 / l
    return 0.0


@pytest.mark.parametrize("frac", [0.2, 0.45, 0.55, 0.8, 0.97])
def test_two_body_closed_form(frac):
    """Two particles: n_i = L (m/rho_j) W'(d) r_hat, n_j = -L (m/rho_i) W'(d) r_hat,
    a_i = K (-gamma m C(d)/d r - gamma (n_i - n_j)), a_j = -a_i."""
    cfg = _cfg()
    l = _f32(cfg["smoothing_length"])
    L = 2.0 * l
    d = frac * L
    x = np.array([[0.5, 0.5, 0.5], [0.5 + d, 0.5, 0.5]], np.float32)
    d = float(np.float64(x[1, 0]) - np.float64(x[0, 0]))  # the distance the oracle sees
    a, s = _tension_dv(x, cfg)
    m = _mass(cfg)
    gam = _f32(GAMMA)
    rho = s.get(O.FIELD_RHO)
    rho_i, rho_j = float(rho[0]), float(rho[1])
    rhat = np.array([-1.0, 0.0, 0.0])  # (x_0 - x_1) / d
    g = _spline_dWdr(d, l)
    n_i = L * (m / rho_j) * g * rhat
    n_j = -L * (m / rho_i) * g * rhat
    K = 2.0 * cfg["rest_density"] / (rho_i + rho_j)
    want = K * (-gam * m * _akinci_C(d, L) / d * (d * rhat) - gam * (n_i - n_j))
    np.testing.assert_allclose(a[0], want, rtol=1e-9, atol=1e-12 * np.abs(want).max())
    np.testing.assert_allclose(a[1], -want, rtol=1e-9, atol=1e-12 * np.abs(want).max())


def test_cohesion_continuous_at_half_support():
    """C's two pieces meet at r = L/2 (pins the L^6/64 term): the two-body
    acceleration is continuous there."""
    cfg = _cfg()
    L = 2.0 * cfg["smoothing_length"]
    out = []
    for eps in (-2e-6, 2e-6):
        x = np.array([[0.5, 0.5, 0.5], [0.5 + 0.5 * L + eps, 0.5, 0.5]], np.float32)
        out.append(_tension_dv(x, cfg)[0][0, 0])
    assert abs(out[0] - out[1]) <= 1e-3 * abs(out[0]), out


def test_cohesion_repels_close_and_attracts_far():
    """With the curvature part taken off (closed-form normals), the cohesion
    pushes a pair apart inside C's root (about 0.27 L) and pulls it together
    beyond."""
    cfg = _cfg()
    L = 2.0 * cfg["smoothing_length"]
    # C < 0 close in (repulsion), C > 0 beyond its root (attraction)
    for frac, attract in ((0.1, False), (0.75, True)):
        x = np.array([[0.5, 0.5, 0.5], [0.5 + frac * L, 0.5, 0.5]], np.float32)
        a, s = _tension_dv(x, cfg)
        m, rho = s.particle_mass(), s.get(O.FIELD_RHO)
        # remove the curvature part using the closed-form normals
        l = cfg["smoothing_length"]
        d = float(np.float64(x[1, 0]) - np.float64(x[0, 0]))
        g = _spline_dWdr(d, l)
        K = 2.0 * cfg["rest_density"] / (rho[0] + rho[1])
        curv = -GAMMA * K * L * g * (m / rho[1] + m / rho[0]) * -1.0
        coh = a[0, 0] - curv
        assert (coh > 0) == attract, (frac, a[0, 0], curv)


def test_momentum_conserved():
    """Every pair term is antisymmetric in (i, j): sum_i a_i = 0."""
    x, _, _, _ = random_box(n=512, seed=3, boundary=False)
    a, _ = _tension_dv(x, _cfg(particle_radius=0.01, smoothing_length=0.02))
    assert np.abs(a).sum() > 0
    assert np.abs(a.sum(0)).max() <= 1e-11 * np.abs(a).sum()


def test_off_and_zero_coefficient_change_nothing():
    x, v, xb, cfg = random_box(n=512, seed=4)
    for over in (dict(enable_surface_tension=False, surface_tension=0.7),
                 dict(enable_surface_tension=True, surface_tension=0.0)):
        c = dict(cfg, **over)
        s = O.Solver(O.config(**c), x, v, xb, O.F32)
        s.density_alpha()
        v0 = s.get(O.FIELD_V)
        s.surface_tension(1e-3)
        assert np.array_equal(s.get(O.FIELD_V), v0), over


def test_binary32_tracks_binary64():
    x, _, _, _ = random_box(n=512, seed=5, boundary=False)
    a64, _ = _tension_dv(x, _cfg(), O.F64)
    a32, _ = _tension_dv(x, _cfg(), O.F32)
    scale = np.abs(a64).max()
    assert np.abs(a32 - a64).max() <= 2e-3 * scale


# --- GPU: the HIP step against the binary32 oracle ----------------------------

def _tension_box(seed, coincident=False, **over):
    x, v, xb, cfg = random_box(n=3000, seed=seed, enable_surface_tension=True,
                               surface_tension=GAMMA, **over)
    if coincident:
        # coincident pairs are left out of the pair lists: these particles
        # take the stencil walk
        x[100] = x[101]
        x[2000] = x[1999]
    return x, v, xb, cfg


@pytest.mark.gpu
@pytest.mark.parametrize("coincident", [False, True])
def test_gpu_tension_step_matches_oracle(coincident):
    x, v, xb, cfg = _tension_box(6, coincident)
    p = Pair(x, v, xb, cfg)
    for k in range(3):
        p.step(1e-3)
        p.compare(f"step {k}")


@pytest.mark.gpu
@pytest.mark.parametrize("n,squeeze", [
    (1, 1.0), (2, 1.0), (63, 1.0), (64, 1.0), (65, 1.0),  # a workgroup holds 64 particles
    (257, 0.75),   # one tile and a particle; lists past the four lanes' first 32 entries
    (1000, 0.45),  # lists past their depth: the stencil walk
])
def test_gpu_tension_edges_match_oracle(n, squeeze):
    x, v, _, cfg = random_box(n=1000, seed=n, boundary=False, enable_surface_tension=True,
                              surface_tension=GAMMA)
    x, v = (0.2 + squeeze * (x[:n] - 0.2)).astype(np.float32), v[:n]
    p = Pair(x, v, None, cfg)
    for k in range(2):
        p.step(2e-4)
        p.compare(f"step {k}")


@pytest.mark.gpu
def test_gpu_tension_changes_the_step():
    x, v, xb, cfg = _tension_box(7)
    on = Pair(x, v, xb, cfg)
    off = Pair(x, v, xb, dict(cfg, enable_surface_tension=False))
    on.gpu.step(1e-3)
    off.gpu.step(1e-3)
    assert not np.array_equal(on.fluid.get_velocities(), off.fluid.get_velocities())


@pytest.mark.gpu
def test_gpu_tension_graph_replay_and_divergence():
    x, v, xb, cfg = _tension_box(8, enable_divergence_solve=True, max_divergence_iters=10)
    p = Pair(x, v, xb, cfg)
    p.gpu.set_graphs(True)
    for k in range(3):
        p.step(1e-3)
        p.compare(f"graph step {k}")


@pytest.mark.gpu
def test_gpu_tension_batched_scenes():
    import water_simulation_amd as ws
    from water_simulation_amd import scenes as SC

    cfg = SC.box_config(max_density_iters=12, enable_surface_tension=True,
                        surface_tension=GAMMA)
    mix = [SC.box_scene(i, n_min=200, n_max=3000) for i in range(3)]
    xb = ws.sample_aabb_boundary((0, 0, 0), (SC.BOX,) * 3, SC.WALL_SPACING, SC.WALL_LAYERS)
    x = np.concatenate([s.positions for s in mix]).astype(np.float32)
    v = np.concatenate([s.velocities for s in mix]).astype(np.float32)
    f = ws.ParticleStore(len(x))
    f.resize(len(x))
    f.set_positions(x)
    f.set_velocities(v)
    b = ws.ParticleStore(len(xb))
    b.resize(len(xb))
    b.set_positions(xb)
    solver = ws.BatchSolver(f, b, ws.DFSPHConfig(**cfg), [len(s.positions) for s in mix],
                            [s.viscosity for s in mix])
    dts = np.array([[1e-3, 8e-4, 1.2e-3], [9e-4, 1e-3, 1.1e-3]], np.float32)
    for dt in dts:
        solver.step(dt)
    for s, sc in enumerate(mix):
        ref = O.Solver(O.config(**dict(cfg, viscosity=sc.viscosity)), sc.positions,
                       sc.velocities, xb, O.F32)
        for dt in dts[:, s]:
            ref.step(float(dt))
        a, e = solver.offsets[s], solver.offsets[s + 1]
        assert_bitexact(f.get_positions()[a:e], ref.get(O.FIELD_X), f"scene {s} position")
        assert_bitexact(f.get_velocities()[a:e], ref.get(O.FIELD_V), f"scene {s} velocity")
        assert solver.scene_stats(s)["density_iters"] == ref.stats()["density_iters"]


@pytest.mark.gpu
def test_gpu_adjoint_refuses_surface_tension():
    from water_simulation_amd import adjoint as A
    from water_simulation_amd._ffi import InvalidArgument

    x, v, xb, cfg = _tension_box(9)
    p = Pair(x, v, xb, cfg)
    g = np.zeros((len(x), 3))
    with pytest.raises(InvalidArgument, match="surface tension"):
        A.adjoint_step(p.gpu, 1e-3, g, g)
    with pytest.raises(InvalidArgument, match="surface tension"):
        A.Rollout(p.gpu, 4)
