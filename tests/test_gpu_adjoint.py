"""The HIP adjoint against the host reference gradient (forward-mode DUAL
oracle along the same binary32 trajectory) and against binary64 central
finite differences with the neighbour structure frozen, for single substeps
(every branch: no iterations, XSPH off, both pressure forms, |v| and domain
clamps) and for checkpointed rollouts, plus the torch.autograd.Function with
the cell-density loss and a viscosity recovery.
"""
from __future__ import annotations

import numpy as np
import pytest

import water_simulation_amd as ws
from water_simulation_amd import adjoint as A
from helpers import random_box
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def make_solver(x, v, xb, cfg):
    n = len(x)
    f = ws.ParticleStore(n)
    f.resize(n)
    f.set_positions(x)
    f.set_velocities(v)
    b = None
    if xb is not None:
        b = ws.ParticleStore(len(xb))
        b.resize(len(xb))
        b.set_positions(xb)
    s = ws.DFSPHSolver(f, b, ws.DFSPHConfig(**cfg))
    s._keep = (f, b)
    return s, f


def dual_directional(x, v, xb, cfg, dts, gx, gv, ux, uv, ue):
    d = O.Solver(O.config(**cfg), x, v, xb, O.DUAL)
    d.seed(dx=ux, dv=uv, d_viscosity=ue)
    for dt in dts:
        d.step(float(dt))
    return float((gx * d.tangent(O.FIELD_X)).sum() + (gv * d.tangent(O.FIELD_V)).sum()), d


def fd_directional(x, v, xb, cfg, dts, gx, gv, ux, uv, ue, eps=1e-6):
    rec = O.Solver(O.config(**cfg), x, v, xb, O.F32)
    tape = O.Tape()
    rec.set_tape(tape, 1)
    for dt in dts:
        rec.step(float(dt))
    val = []
    for sgn in (1.0, -1.0):
        s = O.Solver(O.config(**cfg), x, v, xb, O.F64)
        s.set_state_f64(x.astype(np.float64) + sgn * eps * ux, v.astype(np.float64) + sgn * eps * uv)
        s.set_viscosity_f64(cfg["viscosity"] + sgn * eps * ue)
        s.set_tape(tape, 2)
        for dt in dts:
            s.step(float(dt))
        val.append(float((gx * s.get(O.FIELD_X)).sum() + (gv * s.get(O.FIELD_V)).sum()))
    return (val[0] - val[1]) / (2 * eps)


CASES = {
    "no-iterations": dict(max_density_iters=0, viscosity=0.01),
    "xsph-off": dict(max_density_iters=5, viscosity=0.0),
    "reference-form": dict(max_density_iters=12, viscosity=0.01),
    "kappa-over-rho": dict(max_density_iters=12, viscosity=0.02, pressure_form=1),
    "no-boundary": dict(max_density_iters=6, viscosity=0.01),
}


@pytest.mark.parametrize("case", list(CASES))
def test_adjoint_substep_matches_dual(case):
    over = dict(CASES[case])
    x, v, xb, cfg = random_box(n=343, seed=11, boundary=(case != "no-boundary"), **over)
    dt = 0.002
    rng = np.random.default_rng(3)
    gx = rng.normal(size=x.shape)
    gv = rng.normal(size=x.shape)
    solver, fluid = make_solver(x, v, xb, cfg)
    gxi, gvi, ge = A.adjoint_step(solver, dt, gx, gv)
    assert np.array_equal(fluid.get_positions(), x)  # store back at the input state
    for k in range(3):
        ux = 1e-2 * rng.normal(size=x.shape)
        uv = rng.normal(size=x.shape)
        ue = 0.3 if cfg["viscosity"] > 0 else 0.0
        want, _ = dual_directional(x, v, xb, cfg, [dt], gx, gv, ux, uv, ue)
        got = float((gxi * ux).sum() + (gvi * uv).sum() + ge * ue)
        assert abs(got - want) <= 1e-6 * abs(want), (case, k, got, want)


@pytest.mark.parametrize("n,squeeze", [
    (1, 1.0), (63, 1.0), (65, 0.9),  # a workgroup holds 64 particles
    (257, 0.8),                      # a tile and a particle
    (343, 0.6),                      # lists past their depth: the stencil walk
])
def test_adjoint_of_a_cluster_ignores_a_distant_one(n, squeeze):
    # a second cluster beyond the support moves the first one's working slots
    # (other lanes, workgroups and tiles) and leaves its lists alone: the same bits
    x, v, xb, cfg = random_box(n=343, seed=n, max_density_iters=4, eta_density=0.0)
    a = (0.78 - squeeze * (x[:n] - 0.2)).astype(np.float32)  # beside three walls
    rng = np.random.default_rng(n)
    gx, gv = rng.normal(size=(n + 343, 3)), rng.normal(size=(n + 343, 3))
    one, _ = make_solver(a, v[:n], xb, cfg)
    two, _ = make_solver(np.concatenate([a, x]), np.concatenate([v[:n], v]), xb, cfg)
    wx, wv, _ = A.adjoint_step(one, 2e-4, gx[:n], gv[:n])
    bx, bv, _ = A.adjoint_step(two, 2e-4, gx, gv)
    assert np.abs(wx).max() > 0.0
    assert np.array_equal(bx[:n], wx) and np.array_equal(bv[:n], wv)


def test_adjoint_clamps_match_dual():
    # fast particles (|v| clamp at 5 m/s) next to the walls (domain clamp)
    x, v, xb, cfg = random_box(n=343, seed=4, max_density_iters=4)
    rng = np.random.default_rng(9)
    v = (v + rng.normal(0, 4.0, v.shape)).astype(np.float32)
    x = x.copy()
    # the lowest lattice plane (49 particles, distinct y and z) moved next to
    # x = domain_min + 1e-3 and sent outward
    x[:49, 0] = np.float32(0.0015)
    v[:49, 0] = np.float32(-3.0)
    dt = 0.002
    speed = np.sqrt((v.astype(np.float64) ** 2).sum(1))
    assert (speed > 5.0).sum() > 10
    gx = rng.normal(size=x.shape)
    gv = rng.normal(size=x.shape)
    solver, _ = make_solver(x, v, xb, cfg)
    gxi, gvi, ge = A.adjoint_step(solver, dt, gx, gv)
    for k in range(3):
        ux = 1e-3 * rng.normal(size=x.shape)
        uv = rng.normal(size=x.shape)
        want, _ = dual_directional(x, v, xb, cfg, [dt], gx, gv, ux, uv, 0.2)
        got = float((gxi * ux).sum() + (gvi * uv).sum() + ge * 0.2)
        assert abs(got - want) <= 1e-6 * abs(want), (k, got, want)


def test_rollout_matches_dual_and_fd():
    x, v, xb, cfg = random_box(n=343, seed=21, max_density_iters=8, viscosity=0.02)
    dts = np.full(25, 0.002, np.float32)
    rng = np.random.default_rng(5)
    gx = rng.normal(size=x.shape)
    gv = rng.normal(size=x.shape)
    solver, fluid = make_solver(x, v, xb, cfg)
    ro = A.Rollout(solver, checkpoint_every=7)  # 4 segments, the last partial
    ro.forward(x, v, dts)
    ref = O.Solver(O.config(**cfg), x, v, xb, O.F32)
    for dt in dts:
        ref.step(float(dt))
    assert np.array_equal(fluid.get_positions(), ref.get(O.FIELD_X))
    gx0, gv0, ge = ro.backward(gx, gv)
    for k in range(3):
        ux = 1e-2 * rng.normal(size=x.shape)
        uv = rng.normal(size=x.shape)
        want, _ = dual_directional(x, v, xb, cfg, dts, gx, gv, ux, uv, 0.3)
        got = float((gx0 * ux).sum() + (gv0 * uv).sum() + ge * 0.3)
        assert abs(got - want) <= 1e-6 * abs(want), (k, got, want)
    ux = 1e-2 * rng.normal(size=x.shape)
    uv = rng.normal(size=x.shape)
    fd = fd_directional(x, v, xb, cfg, dts, gx, gv, ux, uv, 0.3)
    got = float((gx0 * ux).sum() + (gv0 * uv).sum() + ge * 0.3)
    assert abs(got - fd) <= 1e-4 * abs(fd), (got, fd)
    print(f"\nrollout: adjoint {got:.9e}  FD(binary64, frozen) {fd:.9e}  rel {abs(got - fd) / abs(fd):.2e}")


def small_inverse(side=8, substeps=40):
    p = A.inverse_problem(side=side, substeps=substeps)
    return p


def test_torch_rollout_density_loss_matches_dual():
    # torch must own the process's HIP runtime, so this runs in a fresh
    # interpreter that imports torch first (see tests/torch_interop.py)
    import json
    import subprocess
    import sys
    from pathlib import Path

    script = Path(__file__).with_name("torch_interop.py")
    r = subprocess.run([sys.executable, "-u", str(script)], capture_output=True, text=True,
                       timeout=240)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    res = json.loads(r.stdout.strip().splitlines()[-1])
    print("\ntorch interop:", res)
    assert res["same_trajectory"]
    assert res["loss_rel_err"] <= 1e-9
    for got, want in res["directional"]:
        assert abs(got - want) <= 1e-5 * abs(want), (got, want)
    assert res["float_viscosity_backward"]
    assert res["stale_tape_refused"]


def test_viscosity_recovery():
    p = small_inverse(side=8, substeps=30)
    cfg = dict(p.cfg, max_density_iters=10, viscosity=0.05)
    solver, fluid = make_solver(p.x0, p.v_true, p.xb, cfg)
    mass = solver.particle_mass()
    ro = A.Rollout(solver, checkpoint_every=10)
    ro.forward(p.x0, p.v_true, p.dts)
    target = A.density_field_np(fluid.get_positions(), mass)
    eps, losses = 0.01, []
    for it in range(12):
        solver.set_viscosity(eps)
        ro.forward(p.x0, p.v_true, p.dts)
        loss, gxl = A.density_loss_np(fluid.get_positions(), target, mass)
        _, _, ge = ro.backward(gxl, np.zeros_like(gxl))
        losses.append(loss)
        # half a Newton step of the quadratic model L = a (eps - eps*)^2, kept in (0, 0.1)
        step = -loss / ge if ge != 0 else 0.0
        eps = float(np.clip(eps + step, 1e-4, 0.1))
    print(f"\nviscosity recovery: losses {losses[0]:.3e} -> {losses[-1]:.3e}, eps {eps:.5f} (true 0.05)")
    assert losses[-1] < 1e-2 * losses[0]
    assert abs(eps - 0.05) < 0.01


def test_inverse_problem_gradient_full_size():
    """The inverse-problem configuration at full size (32^3 particles, 0.6 m
    Akinci box, dt = 0.002 s, checkpoints every 20).  Binary64 central
    differences with the structure frozen along 16 seeded directions over 10
    substeps, and the host reference gradient (forward-mode DUAL oracle along
    the binary32 trajectory) along 4 directions over all 200 substeps, each
    within 1e-3 relative.  The sensitivities of this scene grow ~1.35x per
    substep, through the position dependence of the pressure projection
    (tests/test_oracle_adjoint_growth.py), so the binary64 trajectory that a
    binary64 difference follows separates from the binary32 one the adjoint
    differentiates: max |x64 - x32| is 2e-6 smoothing lengths after 1
    substep, 1.7e-4 after 10 and 0.4 after 20; 10 substeps is the longest
    horizon at which the two still describe the same motion."""
    p = A.inverse_problem(side=32, substeps=200)
    cfg = p.cfg
    solver, fluid = make_solver(p.x0, p.v_guess, p.xb, cfg)
    mass = solver.particle_mass()
    ro = A.Rollout(solver, checkpoint_every=20)
    ro.forward(p.x0, p.v_true, p.dts)
    target = A.density_field_np(fluid.get_positions(), mass)
    rng = np.random.default_rng(2024)
    for horizon, ndir, with_fd in ((10, 16, True), (200, 4, False)):
        dts = p.dts[:horizon]
        tgt = target
        if horizon != 200:
            ro.forward(p.x0, p.v_true, dts)
            tgt = A.density_field_np(fluid.get_positions(), mass)
        ro.forward(p.x0, p.v_guess, dts)
        loss, gxl = A.density_loss_np(fluid.get_positions(), tgt, mass)
        gx0, gv0, ge = ro.backward(gxl, np.zeros_like(gxl))
        got, want = [], []
        for k in range(ndir):
            uv = rng.normal(size=p.x0.shape)
            ue = 0.01 * rng.normal()
            g = float((gv0 * uv).sum() + ge * ue)
            if with_fd:
                w = fd_directional(p.x0, p.v_guess, p.xb, cfg, dts, gxl, np.zeros_like(gxl),
                                   np.zeros_like(uv), uv, ue, eps=1e-7)
            else:
                w, _ = dual_directional(p.x0, p.v_guess, p.xb, cfg, dts, gxl, np.zeros_like(gxl),
                                        np.zeros_like(uv), uv, ue)
            got.append(g)
            want.append(w)
            terms = float(np.abs(gv0 * uv).sum())
            print(f"horizon {horizon} dir {k}: adjoint {g:.6e} reference {w:.6e} "
                  f"rel {abs(g - w) / abs(w):.1e} (sum |terms| / |sum| = {terms / abs(g):.1e})",
                  flush=True)
        got, want = np.array(got), np.array(want)
        # relative error of the gradient projected on the seeded directions (a
        # single direction can be a cancellation residue of its 10^5 terms)
        rel = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"horizon {horizon}: projected-gradient relative error {rel:.2e} "
              f"({'binary64 central differences' if with_fd else 'forward-mode reference'})")
        assert rel <= 1e-3, (horizon, rel)


def test_initial_velocity_recovery():
    """Recover the seeded smooth initial velocity field of an 8^3 block from the
    final cell-density field after 20 substeps by gradient descent with Adam on
    the adjoint gradient: the loss and the velocity error must both fall."""
    p = small_inverse(side=8, substeps=20)
    cfg = dict(p.cfg, max_density_iters=20)
    solver, fluid = make_solver(p.x0, p.v_true, p.xb, cfg)
    mass = solver.particle_mass()
    ro = A.Rollout(solver, checkpoint_every=10)
    ro.forward(p.x0, p.v_true, p.dts)
    target = A.density_field_np(fluid.get_positions(), mass)
    v = p.v_guess.astype(np.float64).copy()
    m1 = np.zeros_like(v)
    m2 = np.zeros_like(v)
    lr, b1, b2 = 0.02, 0.9, 0.999
    err0 = np.linalg.norm(v - p.v_true)
    losses = []
    for it in range(1, 61):
        ro.forward(p.x0, v.astype(np.float32), p.dts)
        loss, gxl = A.density_loss_np(fluid.get_positions(), target, mass)
        _, gv, _ = ro.backward(gxl, np.zeros_like(gxl))
        losses.append(loss)
        m1 = b1 * m1 + (1 - b1) * gv
        m2 = b2 * m2 + (1 - b2) * gv * gv
        v -= lr * (m1 / (1 - b1 ** it)) / (np.sqrt(m2 / (1 - b2 ** it)) + 1e-12)
    err1 = np.linalg.norm(v - p.v_true)
    print(f"\nvelocity recovery: loss {losses[0]:.3e} -> {min(losses):.3e}, "
          f"|v - v_true| {err0:.3f} -> {err1:.3f}")
    assert min(losses) < 0.2 * losses[0]
    assert err1 < err0


def fourier_basis(x: np.ndarray) -> np.ndarray:
    """sin and cos of 2 pi k.x / box for the 27 wave vectors k in {1,2,3}^3:
    the family the inverse problem's smooth velocity fields are drawn from
    (each component of a field is Phi @ c)."""
    xd = x.astype(np.float64) / A.BOX
    cols = []
    for k in [(a, b, c) for a in (1, 2, 3) for b in (1, 2, 3) for c in (1, 2, 3)]:
        arg = 2 * np.pi * (xd * np.array(k)).sum(1)
        cols += [np.sin(arg), np.cos(arg)]
    return np.stack(cols, 1)


def test_initial_velocity_recovery_full_size():
    """Recover the seeded smooth initial velocity field of the full 32^3 block
    from its cell-density field 10 substeps later (the horizon at which the
    binary32 motion is still deterministic to 1e-4 smoothing lengths).  The
    unknowns are the 162 coefficients of the smooth family the field is drawn
    from (a 16^3 density field cannot identify 98,304 per-particle velocities,
    and the divergence-free part of a flow leaves density unchanged); their
    gradient is the adjoint's per-particle gradient chained through the
    basis.  200 Adam steps must cut the loss tenfold and the velocity error
    by 40 %."""
    p = A.inverse_problem(side=32, substeps=10)
    phi = fourier_basis(p.x0)
    coef = lambda v: np.linalg.lstsq(phi, v.astype(np.float64), rcond=None)[0]
    assert np.linalg.norm(phi @ coef(p.v_true) - p.v_true) < 1e-6 * np.linalg.norm(p.v_true)
    c = coef(p.v_guess)
    solver, fluid = make_solver(p.x0, p.v_true, p.xb, p.cfg)
    mass = solver.particle_mass()
    ro = A.Rollout(solver, checkpoint_every=10)
    ro.forward(p.x0, p.v_true, p.dts)
    target = A.density_field_np(fluid.get_positions(), mass)
    vt = p.v_true.astype(np.float64)
    err0 = np.linalg.norm(phi @ c - vt)
    m1, m2 = np.zeros_like(c), np.zeros_like(c)
    lr, b1, b2, iters = 0.02, 0.9, 0.999, 200
    losses = []
    for it in range(1, iters + 1):
        ro.forward(p.x0, (phi @ c).astype(np.float32), p.dts)
        loss, gxl = A.density_loss_np(fluid.get_positions(), target, mass)
        _, gv, _ = ro.backward(gxl, np.zeros_like(gxl))
        losses.append(loss)
        g = phi.T @ gv
        m1 = b1 * m1 + (1 - b1) * g
        m2 = b2 * m2 + (1 - b2) * g * g
        step = lr * 0.5 * (1 + np.cos(np.pi * (it - 1) / iters))
        c = c - step * (m1 / (1 - b1 ** it)) / (np.sqrt(m2 / (1 - b2 ** it)) + 1e-30)
    err1 = np.linalg.norm(phi @ c - vt)
    print(f"\n32^3 velocity recovery over 10 substeps: loss {losses[0]:.3e} -> {min(losses):.3e}, "
          f"|v - v_true| / |v_true| {err0 / np.linalg.norm(vt):.3f} -> {err1 / np.linalg.norm(vt):.3f}")
    assert min(losses) < 0.1 * losses[0]
    assert err1 < 0.6 * err0
