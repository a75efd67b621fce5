"""The mesher's k-NN smoothing where its search plan changes: neighbourhoods
that the guessed radius holds too few or too many points for (surfaces, other
spacings than the particle diameter), equal distances (lattices: lower index
first), coincident points and clumps, every k, against brute force."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import mesh_oracle as M
from test_mesh import _compare

pytestmark = pytest.mark.gpu

R = 0.012


def cloud(case):
    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(*[np.arange(9)] * 3, indexing="ij"), -1).reshape(-1, 3)
    spacing = {"sparse": 5.0 * R, "tight": 0.8 * R}.get(case, 2.0 * R)
    x = 0.1 + spacing * g + (0.0 if case == "lattice" else rng.uniform(-0.2, 0.2, g.shape) * spacing)
    if case == "clump":
        x[:200] = 0.2 + rng.uniform(0.0, 0.3 * R, (200, 3))
        x[200:240] = x[0]  # coincident points
    if case == "sheet":
        x[:, 1] = 0.3
    if case == "lattice":  # exact ties: a power-of-two spacing
        x = 0.125 + g / 64.0
    return x[rng.permutation(len(x))].astype(np.float32)


def brute(pts, k=15, iters=2):
    for _ in range(iters):
        idx = M.knn_brute(pts, k)
        pts = pts[idx].mean(axis=1)
    return pts


@pytest.mark.parametrize("k", [8, 10, 15, 20, 30])
@pytest.mark.parametrize("case", ["fluid", "lattice", "sparse", "tight", "clump", "sheet"])
def test_smoothing_equals_brute_force(case, k, monkeypatch):
    from water_simulation_amd import mesh as WM

    monkeypatch.setattr(M, "smooth_positions_knn", brute)
    x = cloud(case)
    m = WM.SurfaceMesher()
    m.run(x, radius=R, smooth_pre=2, k_neighbors=k)
    _compare(m, M.reconstruct_splat(x, radius=R, smooth_pre=2, k=k), f"{case} k={k}")


def test_more_points_than_one_launch_holds_groups():
    """2,097,152 points fill the launch of the point groups; the rest are taken
    in a second stride (2^29 points would be 2^32 threads, more than a launch
    may hold)."""
    from water_simulation_amd import mesh as WM

    n = 65536 * 32 + 4099
    side = 129
    rng = np.random.default_rng(11)
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (0.1 + 2.0 * R * (g + rng.uniform(-0.2, 0.2, g.shape))).astype(np.float32)
    assert len(x) == n
    m = WM.SurfaceMesher()
    opt = dict(radius=R, smooth_pre=1, smooth_post=0)
    m.run(x, k_neighbors=8, grid_voxel_factor=6.0, smooth_sigma=1.0, **opt)
    _compare(m, M.reconstruct_splat(x, k=8, voxel_factor=6.0, sigma=1.0, **opt), "strided groups")
