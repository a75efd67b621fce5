"""Tiles whose neighbourhood is larger than the staged part of it.

A tile keeps a staging plan up to a second, larger limit: its kernels read the
entries past the staged ones from global memory.  At rest a tile of a block W
particles wide along z has 3 (256 + 2 W) neighbourhood entries: every field
must hold the bits of the kernels that stage nothing, on both sides of both
limits, in both arithmetic modes.  The second limit is above the first from
262,144 working slots in tolerance mode and from 1,048,576 in exact mode.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_bitexact
from test_gpu_lane_shapes import LANES
from test_gpu_quads import DENSE_CFG, ONE_LANE, R, kernel_us, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fast", [False, True], ids=["exact", "fast"])
@pytest.mark.parametrize("dims", [
    (25, 44, 124),   # 1,512 entries: all staged
    (25, 42, 132),   # 1,560: past the staged part
    (22, 15, 420),   # 3,288
    (21, 12, 544),   # 4,032
    (20, 12, 576),   # 4,224
])
def test_wide_tiles_equal_unstaged_kernels(dims, fast):
    rng = np.random.default_rng(dims[2])
    g = np.stack(np.meshgrid(*map(np.arange, dims), indexing="ij"), -1).reshape(-1, 3)
    assert len(g) > 131072  # past every size at which four lanes share a particle
    x = (0.05 + 2 * R * g + rng.uniform(-0.2 * R, 0.2 * R, g.shape)).astype(np.float32)
    v = rng.normal(0.0, 0.4, g.shape).astype(np.float32)
    cfg = dict(rest_density=1000.0, particle_radius=R, smoothing_length=2 * R, viscosity=0.01,
               damping=0.5, domain_min=(0, 0, 0), domain_max=tuple(0.1 + 2 * R * (d + 2) for d in dims),
               max_density_iters=3, enable_divergence_solve=True, max_divergence_iters=2,
               eta_density=1e-6, pressure_form=1, fast_math=fast)
    a, sa = run(x, v, None, cfg, None)
    b, sb = run(x, v, None, cfg, ONE_LANE)
    for k in b:
        assert_bitexact(a[k], b[k], k)
    for k in ("density_iters", "divergence_iters", "mean_density_error", "max_velocity"):
        assert sa[k] == sb[k], (k, sa, sb)


@pytest.mark.parametrize("fast,dims", [
    (False, (68, 66, 236)),   # 2,184 entries
    (False, (46, 43, 544)),   # 4,032: the last plans
    (False, (46, 41, 576)),   # 4,224: most tiles without a plan
    (True, (48, 44, 132)),    # 1,560: a few past the staged ones
    (True, (26, 25, 420)),    # 3,288
    (True, (25, 20, 544)),
    (True, (25, 19, 576)),
])
def test_wide_tiles_of_large_sets_equal_unstaged_kernels(fast, dims):
    rng = np.random.default_rng(dims[2])
    g = np.stack(np.meshgrid(*map(np.arange, dims), indexing="ij"), -1).reshape(-1, 3)
    assert len(g) > (262144 if fast else 1048576)
    x = (0.05 + 2 * R * g + rng.uniform(-0.2 * R, 0.2 * R, g.shape)).astype(np.float32)
    v = rng.normal(0.0, 0.4, g.shape).astype(np.float32)
    cfg = dict(DENSE_CFG, domain_max=tuple(0.1 + 2 * R * (d + 2) for d in dims), max_density_iters=3,
               enable_divergence_solve=True, max_divergence_iters=2, fast_math=fast)
    b, sb = run(x, v, None, cfg, ONE_LANE)
    for shapes in (None, LANES[4]):
        a, sa = run(x, v, None, cfg, shapes)
        for k in b:
            assert_bitexact(a[k], b[k], k)
        for k in ("density_iters", "divergence_iters", "mean_density_error", "max_velocity"):
            assert sa[k] == sb[k], (shapes, k, sa, sb)


@pytest.mark.parametrize("fast", [False, True], ids=["exact", "fast"])
def test_few_wide_tiles_do_not_hold_a_sweep_up(fast):
    """84,800 particles, about one workgroup a CU: a block 40 wide, all of
    whose tiles are staged, and beside it a few rows of 500, whose tiles have
    2,100 to 3,800 entries.  A workgroup that staged a part of those and then
    read the rest from global memory ended the launch late: the sweep took
    1.22 (tolerance mode) and 1.25 times what it takes on the block alone.
    The rows are a tenth of the particles and there is room for them on the
    chip, so half of that is the bound."""
    block = np.stack(np.meshgrid(np.arange(48), np.arange(40), np.arange(40), indexing="ij"), -1)
    rows = np.stack(np.meshgrid(np.arange(51, 55), np.arange(4), np.arange(500), indexing="ij"), -1)
    us = []
    for g in (block.reshape(-1, 3), np.concatenate([block.reshape(-1, 3), rows.reshape(-1, 3)])):
        x = 0.05 + 2 * R * g + np.random.default_rng(5).uniform(-0.2 * R, 0.2 * R, g.shape)
        cfg = dict(DENSE_CFG, domain_max=(1.3, 1.0, 10.2), max_density_iters=20, fast_math=fast)
        us.append(kernel_us(x.astype(np.float32), None, cfg, None, steps=9)["density_change"])
    assert us[1] < 1.11 * us[0], us
