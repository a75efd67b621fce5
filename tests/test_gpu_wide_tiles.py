"""Tiles whose neighbourhood is larger than the staged part of it.

A tile keeps a staging plan up to a second, larger limit: its kernels read the
entries past the staged ones from global memory.  At rest a tile of a block W
particles wide along z has 3 (256 + 2 W) neighbourhood entries: every field
must hold the bits of the kernels that stage nothing, on both sides of both
limits, in both arithmetic modes.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_bitexact
from test_gpu_quads import ONE_LANE, R, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fast", [False, True], ids=["exact", "fast"])
@pytest.mark.parametrize("dims", [
    (25, 44, 124),   # 1,512 entries: all staged
    (25, 42, 132),   # 1,560: a few past the staged ones
    (22, 15, 420),   # 3,288
    (21, 12, 544),   # 4,032: the last plans
    (20, 12, 576),   # 4,224: most tiles without a plan
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
