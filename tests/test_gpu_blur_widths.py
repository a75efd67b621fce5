"""The mesher's blur where its contiguous pass changes: tap radii beyond the
compiled ones (one output per lane on narrow rows, four 64 apart on others),
rows that end before, on and after 64 and 256 columns, against scipy."""
from __future__ import annotations

import time

import numpy as np
import pytest

from oracle import mesh_oracle as M
from test_mesh import _compare

pytestmark = pytest.mark.gpu

R = 0.012


def row(voxels, seed=0):
    """Points whose field is `voxels` wide along the last axis (half a radius each)."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.0, 6.0 * R, (400, 3))
    x[:, 1] = rng.uniform(0.0, 0.5 * R * max(voxels - 16.5, 0.01), 400)  # y: the last axis
    x[0, 1], x[1, 1] = 0.0, 0.5 * R * max(voxels - 16.5, 0.01)
    return x.astype(np.float32)


@pytest.mark.parametrize("sigma", [4.2, 10.0, 16.1])  # R = 17, 40, 64
@pytest.mark.parametrize("width", [17, 63, 64, 65, 128, 256, 257, 320, 321, 600])
def test_wide_blur_equals_scipy(width, sigma):
    from water_simulation_amd import mesh as WM

    opt = dict(radius=R, smooth_pre=0, smooth_post=0)
    x = row(width)
    m = WM.SurfaceMesher()
    info = m.run(x, smooth_sigma=sigma, **opt)
    assert info["dims"][2] == width
    _compare(m, M.reconstruct_splat(x, sigma=sigma, **opt), f"width {width} sigma {sigma}")


def test_wide_blur_of_a_thin_field_costs_its_taps():
    """A field of 1,202 x 1,203 x 17 voxels: 81 taps take at most one and a half
    times the run with 29 (2.2 times while a lane's outputs lay side by side)."""
    from water_simulation_amd import mesh as WM

    rng = np.random.default_rng(0)
    g = np.stack(np.meshgrid(np.arange(300), np.arange(300), indexing="ij"), -1).reshape(-1, 2)
    x = np.full((len(g), 3), 0.1)
    x[:, [0, 2]] += 2 * R * (g + rng.uniform(-0.2, 0.2, g.shape))
    x = x.astype(np.float32)
    ms = {}
    for sigma in (3.5, 10.0):
        m = WM.SurfaceMesher()
        t = []
        for _ in range(7):
            t0 = time.perf_counter()
            m.run(x, radius=R, smooth_sigma=sigma)
            t.append(1e3 * (time.perf_counter() - t0))
        ms[sigma] = float(np.median(t[2:]))
    print(ms)
    assert ms[10.0] < 1.5 * ms[3.5]
