"""One and four lanes per particle as launch shapes.

The default shapes choose between them by the size of the working set; the
values 1 and 4 take either at any size.  Small scenes then reach the staged
kernels of large ones and the reverse: both against the binary32 oracle where
the default kernels are, and against the kernels that stage nothing where the
lists overflow or tiles have no staging plan.
"""
from __future__ import annotations

import numpy as np
import pytest

import water_simulation_amd as ws
from water_simulation_amd import scenes as SC
from helpers import Pair, assert_bitexact, random_box
from oracle import oracle as O
from test_gpu_batch import Batch, run_plain, wall_positions
from test_gpu_quads import DENSE_CFG, ONE_LANE, R, cloud, kernel_us, pile, run

pytestmark = pytest.mark.gpu

LANES = {k: dict(density_alpha_nt=k, xsph_nt=k, change_nt=k, apply_nt=k) for k in (1, 4)}


@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("over", [
    dict(),
    dict(pressure_form=1, enable_divergence_solve=True, max_divergence_iters=5),
    dict(escape=True),
], ids=["plain", "divergence", "escapees"])
def test_small_scenes_match_oracle(over, lanes):
    over = dict(over)
    escape = over.pop("escape", False)
    x, v, xb, cfg = random_box(n=1000, seed=21, **over)
    if escape:  # tiles without a staging plan, the speed and the domain clamp
        x[:8] = [[-0.5, 0.1, 0.1], [2.0, 0.1, 0.1], [0.1, -3.0, 0.1], [0.1, 9.0, 0.1],
                 [0.1, 0.1, -1.0], [0.1, 0.1, 4.0], [-1.0, -1.0, -1.0], [1e6, 1e6, 1e6]]
        v[8:40] *= 40.0
    p = Pair(x, v, xb, cfg)
    p.gpu.set_shapes(**LANES[lanes])
    for k in range(3):
        p.step(5e-4)
        p.compare(f"{lanes} lanes step {k}")


def scene(case, n):
    """Clumps over the list depth, coincident pairs, escapees; `wide` is past
    the staged part of a tile, with a squeezed corner (n layers; tiles of such
    neighbourhoods have plans from 48 layers on in tolerance mode, 182 in exact
    mode, and gather everything below)."""
    if case == "wide":
        dims = (n, 44, 132)
        g = np.stack(np.meshgrid(*map(np.arange, dims), indexing="ij"), -1).reshape(-1, 3)
        rng = np.random.default_rng(n)
        x = 0.05 + 2 * R * g + rng.uniform(-0.2 * R, 0.2 * R, g.shape)
        c = (g < 12).all(1)
        x[c] = 0.05 + 0.6 * (x[c] - 0.05)
        x = x.astype(np.float32)
        v = rng.normal(0.0, 0.4, x.shape).astype(np.float32)
    else:
        x, v = cloud(n, True)
        x[n // 2 : n // 2 + 150] = pile(150) * 0.8
    x[7] = x[8]
    x[40:43] = [[-5.0, 0.2, 0.2], [np.nan, 0.2, 0.2], [0.2, 0.2, 90.0]]
    return x, v


@pytest.mark.parametrize("fast", [False, True], ids=["exact", "fast"])
@pytest.mark.parametrize("case,n,lanes", [
    ("clump", 300, 1), ("clump", 4000, 1), ("clump", 4000, 4),
    ("clump", 140000, None), ("clump", 140000, 4),  # None: the default, one lane at this size
    ("wide", 24, None), ("wide", 24, 4), ("wide", 48, None), ("wide", 48, 4),
    ("wide", 182, None), ("wide", 182, 4),
])
def test_irregular_scenes_equal_unstaged_kernels(case, n, lanes, fast):
    x, v = scene(case, n)
    hi = tuple(float(np.ceil(np.nanmax(x[100:, a]) + 0.1)) for a in range(3))
    cfg = dict(DENSE_CFG, domain_max=hi, max_density_iters=3, enable_divergence_solve=True,
               max_divergence_iters=2, fast_math=fast)
    xb = O.sample_aabb_boundary([0, 0, 0], hi, 2 * R, 2) if case == "clump" else None
    a, sa = run(x, v, xb, cfg, LANES.get(lanes))
    b, sb = run(x, v, xb, cfg, ONE_LANE)
    for k in b:
        assert_bitexact(a[k], b[k], k)
    for k in ("density_iters", "divergence_iters", "mean_density_error", "nan_count"):
        assert sa[k] == sb[k], (k, sa, sb)


@pytest.mark.parametrize("lanes", [1, 4])
def test_uneven_batch_with_empty_scenes(lanes):
    xb = wall_positions()
    cfg = SC.box_config(max_density_iters=10)
    mix = [SC.box_scene(s, n_min=a, n_max=a + 1) for s, a in enumerate((1, 300, 64, 2100))]
    for empty in (0, 3):
        s = SC.box_scene(50 + empty, n_min=10, n_max=11)
        s.positions, s.velocities = s.positions[:0], s.velocities[:0]
        mix.insert(empty, s)
    b = Batch(mix, xb, cfg)
    b.solver.set_shapes(**LANES[lanes])
    for _ in range(2):
        b.step()
    for s, m in enumerate(mix):
        if not len(m.positions):
            continue
        want, _ = run_plain(m, xb, cfg, np.array(b.dts)[:, s], shapes=ONE_LANE)
        got = b.scene(s)
        for k in got:
            assert_bitexact(got[k], want[k], f"{lanes} lanes, scene {s}, {k}")


def test_shape_values_are_checked_and_kept():
    x, v = cloud(200, False)
    f = ws.ParticleStore(200)
    f.resize(200)
    f.set_positions(x)
    f.set_velocities(v)
    s = ws.DFSPHSolver(f, None, ws.DFSPHConfig(**DENSE_CFG))
    default = s.shapes()
    assert (default["density_alpha_nt"], default["xsph_nt"], default["change_nt"],
            default["apply_nt"]) == (256, 0, 0, 0)
    for k, shapes in LANES.items():
        s.set_shapes(**shapes)
        assert {n: s.shapes()[n] for n in shapes} == shapes
    for name in LANES[1]:
        with pytest.raises(ValueError):
            s.set_shapes(**{name: 2})
    with pytest.raises(ValueError):
        s.set_shapes(density_alpha_nt=0)
    # the autotuner times both and names the one it keeps
    s.step(1e-4)
    log = s.autotune(reps=1)
    for kernel in ("density_alpha", "xsph", "density_change", "apply_kappa"):
        assert {1, 4} <= {r[1] for r in log if r[0] == kernel}, kernel
    assert 0 not in (s.shapes()["xsph_nt"], s.shapes()["change_nt"], s.shapes()["apply_nt"])
    s.step(1e-4)


def test_density_of_an_open_block_takes_the_faster_kernel():
    """98,304 particles without a boundary, tolerance mode: four lanes take 1.12
    to 1.15 times as long as one."""
    g = np.stack(np.meshgrid(np.arange(48), np.arange(32), np.arange(64), indexing="ij"), -1)
    g = g.reshape(-1, 3)
    x = (0.06 + 2 * R * (g + np.random.default_rng(0).uniform(-0.1, 0.1, g.shape))).astype(np.float32)
    cfg = dict(DENSE_CFG, domain_max=(1.1, 0.8, 1.5), fast_math=True)
    t = {k: kernel_us(x, None, cfg, s, steps=25)["density_alpha"]
         for k, s in (("default", None), (1, LANES[1]), (4, LANES[4]))}
    print(t)
    assert t["default"] < 1.08 * min(t[1], t[4])
