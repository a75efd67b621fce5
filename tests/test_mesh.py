"""Surface meshes from particle frames (the splat method of
tools/particles_to_mesh.py:77-138 on the GPU).

CPU: the oracle is pinned -- its blur restatement equals
scipy.ndimage.gaussian_filter bit for bit (the GPU computes that
restatement), the marching-cubes table closes every surface, orients it
outwards, and gives a sphere's area and volume and the Euler characteristic
of a sphere and a torus; the library's table equals the oracle's.
GPU: grid set-up, splat, blur, iso level, vertices and triangles of the HIP
path equal the oracle bit for bit (and the blurred grid equals scipy's).
"""
from __future__ import annotations

from collections import Counter

import numpy as np
import pytest
import scipy.ndimage

from oracle import mesh_oracle as M


def _mesh_checks(v, t):
    """(closed and consistently oriented, Euler characteristic, area, volume)."""
    d = Counter()
    for a, b, c in t:
        for x, y in ((a, b), (b, c), (c, a)):
            d[(int(x), int(y))] += 1
    closed = all(d[(y, x)] == n for (x, y), n in d.items())
    E = len({tuple(sorted(k)) for k in d})
    V = len(np.unique(t))
    p = v.astype(np.float64)
    a, b, c = p[t[:, 0]], p[t[:, 1]], p[t[:, 2]]
    area = 0.5 * np.linalg.norm(np.cross(b - a, c - a), axis=1).sum()
    vol = np.einsum("ij,ij->i", a, np.cross(b, c)).sum() / 6.0
    return closed, V - E + len(t), area, vol


def _centered(n):
    x = np.arange(n) - (n - 1) / 2
    return np.meshgrid(x, x, x, indexing="ij")


def test_blur_restatement_is_scipy():
    rng = np.random.default_rng(0)
    for shape, sigma in (((8, 9, 10), 2.5), ((20, 13, 31), 2.5), ((11, 12, 9), 1.3)):
        g = rng.integers(0, 5, shape).astype(np.float32)
        got = M.blur_restated(g, sigma)
        want = scipy.ndimage.gaussian_filter(g, sigma=sigma)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (shape, sigma)


def test_sphere_closed_outward_area_volume():
    n, R = 48, 15.3
    X, Y, Z = _centered(n)
    g = (R - np.sqrt(X ** 2 + Y ** 2 + Z ** 2)).astype(np.float32)
    v, t = M.marching_cubes(g, np.float32(0.0), -np.full(3, (n - 1) / 2), np.ones(3))
    closed, chi, area, vol = _mesh_checks(v, t)
    assert closed and chi == 2
    assert abs(area / (4 * np.pi * R ** 2) - 1) < 0.01
    assert abs(vol / (4 / 3 * np.pi * R ** 3) - 1) < 0.01  # positive: normals point outwards


def test_torus_euler_characteristic():
    n = 40
    X, Y, Z = _centered(n)
    q = np.sqrt(X ** 2 + Y ** 2) - 11.0
    g = (4.5 - np.sqrt(q ** 2 + Z ** 2)).astype(np.float32)
    v, t = M.marching_cubes(g, np.float32(0.0), np.zeros(3), np.ones(3))
    closed, chi, _, vol = _mesh_checks(v, t)
    assert closed and chi == 0 and vol > 0


def test_random_fields_closed():
    for seed in range(3):
        g = np.random.default_rng(seed).random((12, 11, 13)).astype(np.float32)
        g[[0, -1]] = 0
        g[:, [0, -1]] = 0
        g[:, :, [0, -1]] = 0
        v, t = M.marching_cubes(g, np.float32(0.5), np.zeros(3), np.ones(3))
        closed, _, _, vol = _mesh_checks(v, t)
        assert closed and vol > 0, seed


def test_complementary_configurations_cut_the_same_edges():
    counts, tris = M.table()
    for cfg in range(256):
        a = set(tris[cfg, :3 * counts[cfg]].tolist())
        b = set(tris[255 - cfg, :3 * counts[255 - cfg]].tolist())
        assert a == b, cfg
        # the edges cut are exactly those between an inside and an outside corner
        cut = set()
        for c0 in range(8):
            for ax in range(3):
                c1 = c0 | (1 << ax)
                if c1 != c0 and ((cfg >> c0) & 1) != ((cfg >> c1) & 1):
                    cut.add(M._edge(c0, c1))
        assert a == cut, cfg


def _grid_mesh(n=6, z=None):
    """A triangulated n x n vertex grid in the plane z = 0 (or height z(x, y))."""
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    v = np.stack([i.ravel(), j.ravel(), np.zeros(n * n)], 1).astype(np.float32)
    if z is not None:
        v[:, 2] = z(v[:, 0], v[:, 1])
    t = []
    for a in range(n - 1):
        for b in range(n - 1):
            p = a * n + b
            t += [(p, p + n, p + n + 1), (p, p + n + 1, p + 1)]
    return v, np.array(t, np.uint32)


def test_laplacian_neighbours_come_from_triangles():
    t = np.array([[0, 1, 2], [0, 2, 3], [0, 3, 1], [1, 3, 2]], np.uint32)  # a tetrahedron
    table, valid = M.vertex_neighbours(t, 4)
    for v in range(4):
        assert table[v][valid[v]].tolist() == [u for u in range(4) if u != v]


def test_laplacian_step_is_half_way_to_inverse_distance_mean():
    """A fan around vertex 0 with neighbours at distances 1, 2, 4: weights
    1, 1/2, 1/4 (inverse distance, not squared, not uniform), lambda 0.5."""
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 2, 0], [0, 0, 4]], np.float32)
    t = np.array([[0, 1, 2], [0, 2, 3], [0, 3, 1]], np.uint32)
    out = M.laplacian_smooth(v, t, 1)
    mean = (1.0 * v[1] + 0.5 * v[2] + 0.25 * v[3]) / 1.75
    assert np.allclose(out[0], 0.5 * mean, rtol=1e-6, atol=1e-9)
    # every vertex reads the previous pass (not vertex 0's new position):
    # vertex 1 sees 0, 2, 3 at distances 1, sqrt 5, sqrt 17
    w = np.array([1.0, 1 / np.sqrt(5.0), 1 / np.sqrt(17.0)])
    mean1 = (w[0] * v[0] + w[1] * v[2] + w[2] * v[3]) / w.sum()
    assert np.allclose(out[1], v[1] + 0.5 * (mean1 - v[1]), rtol=1e-6, atol=1e-9)


def test_laplacian_keeps_planes_and_symmetric_vertices():
    v, t = _grid_mesh(7)
    out = M.laplacian_smooth(v, t, 3)
    assert np.all(out[:, 2] == 0)
    # an interior vertex of the regular grid has its neighbours in symmetric pairs
    assert np.allclose(out[3 * 7 + 3], v[3 * 7 + 3], atol=1e-6)
    # a bump flattens
    vb, tb = _grid_mesh(7, z=lambda x, y: np.where((x == 3) & (y == 3), 1.0, 0.0))
    ob = M.laplacian_smooth(vb, tb, 1)
    assert 0 < ob[3 * 7 + 3, 2] < 1


def test_laplacian_shrinks_a_sphere_slightly():
    n, R = 48, 15.0
    X, Y, Z = _centered(n)
    g = (R - np.sqrt(X ** 2 + Y ** 2 + Z ** 2)).astype(np.float32)
    v, t = M.marching_cubes(g, np.float32(0.0), np.zeros(3), np.ones(3))
    c = np.array([(n - 1) / 2] * 3)
    r0 = np.linalg.norm(v - c, axis=1).mean()
    s = M.laplacian_smooth(v, t, 2)
    r2 = np.linalg.norm(s - c, axis=1).mean()
    assert r2 < r0 and r0 - r2 < 0.02 * R
    assert _mesh_checks(s, t)[0]


def test_ckdtree_neighbours_are_brute_force_order():
    """On points without distance ties, cKDTree.query's rows are the k
    nearest in ascending distance, self first: the order the GPU sums in."""
    from scipy.spatial import cKDTree

    rng = np.random.default_rng(7)
    x = rng.uniform(0, 1, (400, 3))
    _, idx = cKDTree(x).query(x, k=15)
    assert np.array_equal(idx, M.knn_brute(x, 15))
    assert np.array_equal(idx[:, 0], np.arange(len(x)))


def test_knn_smoothing_pulls_points_together():
    """Each pass replaces a point by a mean of neighbours: the cloud's spread
    shrinks, its mean stays within the hull, a lattice interior is a fixed
    point of one pass up to rounding."""
    rng = np.random.default_rng(8)
    x = rng.normal(0, 1, (300, 3))
    y = M.smooth_positions_knn(x, k=10, iters=1)
    assert y.std(0).max() < x.std(0).max()
    g = np.stack(np.meshgrid(*[np.arange(9.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
    s = M.smooth_positions_knn(g, k=7, iters=1)
    inner = np.all((g >= 2) & (g <= 6), axis=1)
    assert np.abs(s[inner] - g[inner]).max() < 1e-12  # self + 6 face neighbours


def test_library_table_is_the_oracles():
    from water_simulation_amd import mesh as WM

    c, e = WM.mc_table()
    oc, oe = M.table()
    assert np.array_equal(c, oc) and np.array_equal(e, oe)


# ---- GPU ---------------------------------------------------------------------

def _cloud(seed=0, n_side=24, r=0.012):
    rng = np.random.default_rng(seed)
    i = np.arange(n_side, dtype=np.float32)
    g = np.stack(np.meshgrid(i, i, i, indexing="ij"), -1).reshape(-1, 3)
    x = np.float32(0.1) + np.float32(2 * r) * g
    x += rng.uniform(-0.3 * r, 0.3 * r, x.shape).astype(np.float32)
    # a splash above the block
    s = rng.normal([0.4, 0.8, 0.35], 0.03, (300, 3)).astype(np.float32)
    return np.concatenate([x, s]).astype(np.float32)


def _compare(mesher, want, tag):
    info = mesher.info()
    assert tuple(info["dims"]) == tuple(int(k) for k in want["res"]), tag
    assert np.array_equal(info["lo"], want["lo"]) and np.array_equal(info["extent"],
                                                                      want["extent"]), tag
    g = mesher.grid()
    assert np.array_equal(g.view(np.uint32), want["grid"].view(np.uint32)), tag
    assert info["iso"].view(np.uint32) == np.float32(want["iso"]).view(np.uint32), tag
    v, t = mesher.vertices(), mesher.triangles()
    assert v.shape == want["vertices"].shape and t.shape == want["triangles"].shape, tag
    assert np.array_equal(v.view(np.uint32), want["vertices"].view(np.uint32)), tag
    assert np.array_equal(t, want["triangles"]), tag
    return v, t


@pytest.mark.gpu
@pytest.mark.parametrize("swap", [True, False])
def test_gpu_mesh_matches_oracle(swap):
    from water_simulation_amd import mesh as WM

    x = _cloud(1)
    m = WM.SurfaceMesher()
    m.run(x, radius=0.012, swap_yz=swap)
    want = M.reconstruct_splat(x, radius=0.012, swap_yz=swap)
    v, t = _compare(m, want, f"swap {swap}")
    closed, _, _, vol = _mesh_checks(v, t)
    assert closed and vol > 0


@pytest.mark.gpu
def test_gpu_mesh_options_and_store_input():
    import water_simulation_amd as ws
    from water_simulation_amd import mesh as WM

    x = _cloud(2, n_side=16, r=0.01)
    st = ws.ParticleStore(len(x))
    st.resize(len(x))
    st.set_positions(x)
    m = WM.SurfaceMesher()
    for kw in (dict(smooth_sigma=0.0), dict(grid_voxel_factor=0.8, smooth_sigma=1.5,
                                           iso_factor=0.3)):
        m.run(st, radius=0.01, **kw)
        want = M.reconstruct_splat(x, radius=0.01, voxel_factor=kw.get("grid_voxel_factor", 0.5),
                                   sigma=kw["smooth_sigma"], iso_factor=kw.get("iso_factor", 0.18))
        _compare(m, want, str(kw))


@pytest.mark.gpu
def test_gpu_mesh_cli_writes_ply(tmp_path):
    import water_simulation_amd as ws
    from water_simulation_amd import mesh as WM

    x = _cloud(3, n_side=12)
    ws.write_frame(str(tmp_path / "frame_0001.bin"), x)
    ws.write_frame(str(tmp_path / "frame_0002.bin"), x[::-1].copy())
    assert WM.main(["--seq", str(tmp_path), "--out-dir", str(tmp_path / "mesh")]) == 0
    for k in (1, 2):
        data = (tmp_path / "mesh" / f"frame_000{k}.ply").read_bytes()
        head, _, body = data.partition(b"end_header\n")
        nv = int(head.split(b"element vertex ")[1].split(b"\n")[0])
        nf = int(head.split(b"element face ")[1].split(b"\n")[0])
        assert len(body) == 12 * nv + 13 * nf and nf > 0
    # --smooth 0: the Laplacian passes off; vertex and face counts do not change
    assert WM.main(["--frame", str(tmp_path / "frame_0001.bin"), "--out", str(tmp_path / "a.ply"),
                    "--smooth", "0"]) == 0
    assert (tmp_path / "a.ply").read_bytes()[:200].split(b"end_header")[0] == \
        (tmp_path / "mesh" / "frame_0001.ply").read_bytes()[:200].split(b"end_header")[0]


@pytest.mark.gpu
def test_gpu_mesh_frame_cpp_app_matches_python(tmp_path):
    """bin/mesh_frame (the C++ water::SurfaceMesher over a ParticleStore,
    default weights computed by the library in scipy's order) writes the
    same PLY bytes as the Python command line; its flags reach the mesher."""
    import subprocess
    from pathlib import Path

    import water_simulation_amd as ws
    from water_simulation_amd import mesh as WM

    app = Path(__file__).resolve().parents[1] / "water_simulation_amd" / "bin" / "mesh_frame"
    assert app.exists(), "mesh_frame is not built"
    x = _cloud(9, n_side=12)
    f = tmp_path / "frame_0001.bin"
    ws.write_frame(str(f), x)
    r = subprocess.run([str(app), "--frame", str(f), "--out", str(tmp_path / "cpp.ply")],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert WM.main(["--frame", str(f), "--out", str(tmp_path / "py.ply")]) == 0
    assert (tmp_path / "cpp.ply").read_bytes() == (tmp_path / "py.ply").read_bytes()
    r = subprocess.run([str(app), "--frame", str(f), "--out", str(tmp_path / "cpp2.ply"),
                        "--smooth", "0", "--smooth-pre", "1", "--k-neighbors", "8", "--no-swap",
                        "--iso-factor", "0.3"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    m = WM.SurfaceMesher()
    m.run(x, smooth_post=0, smooth_pre=1, k_neighbors=8, swap_yz=False, iso_factor=0.3)
    WM.write_ply(tmp_path / "py2.ply", m.vertices(), m.triangles())
    assert (tmp_path / "cpp2.ply").read_bytes() == (tmp_path / "py2.ply").read_bytes()
    r = subprocess.run([str(app), "--frame", str(f), "--out", str(tmp_path / "bad.ply"),
                        "--k-neighbors", "7"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 1 and "k_neighbors" in r.stderr


@pytest.mark.gpu
def test_gpu_library_weights_use_numpy_sum_order(tmp_path):
    """sigma 3: the C library's exp equals numpy's on every tap, but the
    normalised weights differ between a sequential sum and numpy's pairwise
    sum, so mesh_frame (library weights) matches the Python command line
    (numpy weights) byte for byte only if the library sums in numpy's order."""
    import math
    import subprocess
    from pathlib import Path

    import water_simulation_amd as ws
    from water_simulation_amd import mesh as WM

    sigma = 3.0
    R = int(4 * sigma + 0.5)
    arg = -0.5 / (sigma * sigma) * np.arange(-R, R + 1) ** 2
    phi = np.exp(arg)
    if not np.array_equal(phi, np.array([math.exp(v) for v in arg])):
        pytest.skip("this machine's numpy exp differs from the C library's at sigma 3")
    seq = 0.0
    for v in phi:
        seq = seq + v
    assert not np.array_equal(phi / phi.sum(), phi / seq)  # the order matters here
    app = Path(__file__).resolve().parents[1] / "water_simulation_amd" / "bin" / "mesh_frame"
    x = _cloud(10, n_side=12)
    f = tmp_path / "frame_0001.bin"
    ws.write_frame(str(f), x)
    r = subprocess.run([str(app), "--frame", str(f), "--out", str(tmp_path / "cpp.ply"),
                        "--smooth-sigma", "3"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert WM.main(["--frame", str(f), "--out", str(tmp_path / "py.ply"),
                    "--smooth-sigma", "3"]) == 0
    assert (tmp_path / "cpp.ply").read_bytes() == (tmp_path / "py.ply").read_bytes()


@pytest.mark.gpu
def test_gpu_mesh_rejects_empty():
    from water_simulation_amd import mesh as WM
    from water_simulation_amd._ffi import InvalidArgument

    with pytest.raises(InvalidArgument):
        WM.SurfaceMesher().run(np.zeros((0, 3), np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("pre", [2, 0])
def test_gpu_mesh_rejects_non_finite_points(bad, pre):
    """One non-finite coordinate among finite points: the bounds pass counts
    it (min/max skip NaN) and the host refuses the set before any k-NN search
    or splat runs."""
    from water_simulation_amd import mesh as WM
    from water_simulation_amd._ffi import InvalidArgument

    pts = _cloud(3, n_side=6)
    pts[17, 1] = bad
    with pytest.raises(InvalidArgument):
        WM.SurfaceMesher().run(pts, smooth_pre=pre)


@pytest.mark.gpu
def test_gpu_mesh_of_a_solver_store_after_steps():
    """The consumer downstream of the solver: mesh the store's device
    positions after a few substeps, against the oracle on the same frame."""
    import water_simulation_amd as ws
    from water_simulation_amd import mesh as WM
    from helpers import random_box

    x, v, xb, cfg = random_box(n=3000, seed=11)
    f = ws.ParticleStore(len(x))
    f.resize(len(x))
    f.set_positions(x)
    f.set_velocities(v)
    b = ws.ParticleStore(len(xb))
    b.resize(len(xb))
    b.set_positions(xb)
    s = ws.DFSPHSolver(f, b, ws.DFSPHConfig(**cfg))
    for _ in range(3):
        s.step(1e-3)
    m = WM.SurfaceMesher()
    m.run(f, radius=cfg["particle_radius"])
    want = M.reconstruct_splat(f.get_positions(), radius=cfg["particle_radius"])
    v_, t_ = _compare(m, want, "solver store")
    assert len(t_) > 0 and _mesh_checks(v_, t_)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["one point", "identical points", "wide blur", "widest blur",
                                  "no surface"])
def test_gpu_mesh_edge_cases(case):
    from water_simulation_amd import mesh as WM

    kw = dict(radius=0.01)
    if case == "one point":  # fewer points than k: no position smoothing
        x = np.array([[0.3, 0.2, 0.1]], np.float32)
        kw.update(smooth_pre=0)
    elif case == "identical points":  # all distances tie: no position smoothing
        x = np.tile(np.array([[0.5, 0.5, 0.5]], np.float32), (50, 1))
        kw.update(smooth_pre=0)
    elif case == "wide blur":  # 41 taps on an 8-voxel minimum grid: reflections wrap
        x = np.random.default_rng(4).uniform(0.0, 0.01, (40, 3)).astype(np.float32)
        kw.update(smooth_sigma=5.0, grid_voxel_factor=4.0)
    elif case == "widest blur":  # 137 taps: more than the tiled passes stage, one load per tap
        x = np.random.default_rng(5).uniform(0.0, 0.01, (40, 3)).astype(np.float32)
        kw.update(smooth_sigma=17.0, grid_voxel_factor=4.0)
    else:  # the iso level above the maximum: no crossing edge
        x = _cloud(5, n_side=6)
        kw.update(iso_factor=1.5)
    m = WM.SurfaceMesher()
    m.run(x, **kw)
    want = M.reconstruct_splat(x, radius=kw["radius"], voxel_factor=kw.get("grid_voxel_factor", 0.5),
                               sigma=kw.get("smooth_sigma", 2.5), iso_factor=kw.get("iso_factor", 0.18),
                               smooth_pre=kw.get("smooth_pre", 2))
    v, t = _compare(m, want, case)
    if case == "no surface":
        assert len(v) == 0 and len(t) == 0
    else:
        assert _mesh_checks(v, t)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("k,iters", [(8, 1), (15, 3), (30, 2)])
def test_gpu_knn_smoothing_matches_ckdtree(k, iters):
    from water_simulation_amd import mesh as WM

    x = _cloud(6, n_side=14)
    m = WM.SurfaceMesher()
    m.run(x, radius=0.012, smooth_pre=iters, k_neighbors=k)
    _compare(m, M.reconstruct_splat(x, radius=0.012, smooth_pre=iters, k=k), f"k={k} x{iters}")


@pytest.mark.gpu
@pytest.mark.parametrize("k,iters", [(15, 2), (30, 1)])
def test_gpu_knn_smoothing_isolated_points(k, iters):
    """Points far from the rest (tens of 4r cells away) are searched by the
    wave-per-point pass after the per-point ring walk gives up."""
    from water_simulation_amd import mesh as WM

    rng = np.random.default_rng(11)
    far = (np.float32(0.1) + rng.uniform(0.5, 1.5, (12, 3))).astype(np.float32)
    x = np.concatenate([_cloud(7, n_side=10), far]).astype(np.float32)
    m = WM.SurfaceMesher()
    m.run(x, radius=0.012, smooth_pre=iters, k_neighbors=k)
    _compare(m, M.reconstruct_splat(x, radius=0.012, smooth_pre=iters, k=k),
             f"isolated k={k} x{iters}")


@pytest.mark.gpu
@pytest.mark.parametrize("post", [0, 1, 3])
def test_gpu_laplacian_smoothing_matches_oracle(post):
    from water_simulation_amd import mesh as WM

    x = _cloud(8, n_side=14)
    m = WM.SurfaceMesher()
    m.run(x, radius=0.012, smooth_post=post)
    _compare(m, M.reconstruct_splat(x, radius=0.012, smooth_post=post), f"post={post}")


@pytest.mark.gpu
def test_gpu_knn_smoothing_points_on_a_line():
    """A thin grid (one cell across) with uneven gaps: many points need far
    more than three rings, searched row by row within the grid."""
    from water_simulation_amd import mesh as WM

    rng = np.random.default_rng(12)
    xs = np.float32(0.1) + np.cumsum(rng.uniform(0.002, 0.2, 150)).astype(np.float32)
    x = np.stack([xs, np.full(150, 0.3, np.float32), np.full(150, 0.2, np.float32)], 1)
    m = WM.SurfaceMesher()
    m.run(x, radius=0.012, smooth_pre=2, k_neighbors=8)
    _compare(m, M.reconstruct_splat(x, radius=0.012, smooth_pre=2, k=8), "line")


@pytest.mark.gpu
def test_gpu_knn_smoothing_rejects_bad_k():
    from water_simulation_amd import mesh as WM
    from water_simulation_amd._ffi import InvalidArgument

    m = WM.SurfaceMesher()
    with pytest.raises(InvalidArgument):
        m.run(_cloud(1, n_side=4), k_neighbors=7)
    with pytest.raises(InvalidArgument):
        m.run(np.zeros((10, 3), np.float32), k_neighbors=15)


@pytest.mark.gpu
def test_gpu_mesher_keeps_nothing_of_other_frames():
    """One mesher on a small, a large and again a small frame with other blurs,
    neighbour counts and smoothings: each equals the oracle."""
    from water_simulation_amd import mesh as WM

    rng = np.random.default_rng(9)
    r = 0.012

    def frame(n, wide):
        g = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)
        x = 0.1 + 2 * r * (g + rng.uniform(-0.3, 0.3, g.shape))
        if wide:  # spray far above: a box mostly empty
            x = np.concatenate([x, rng.uniform(0.0, 1.5, (60, 3))])
        return x.astype(np.float32)

    m = WM.SurfaceMesher()
    for k, (n, wide, o) in enumerate([
        (6, False, dict()),
        (14, False, dict(sigma=4.2, k=8, smooth_post=5)),
        (7, True, dict(sigma=1.0, k=30, smooth_pre=1)),
        (5, False, dict(sigma=0.0, smooth_pre=0, smooth_post=0)),
        (12, True, dict(sigma=3.0, smooth_pre=3, smooth_post=0)),
        (6, False, dict()),
    ]):
        x = frame(n, wide)
        names = dict(sigma="smooth_sigma", k="k_neighbors")
        m.run(x, radius=r, **{names.get(a, a): b for a, b in o.items()})
        _compare(m, M.reconstruct_splat(x, radius=r, **o), f"frame {k}")


@pytest.mark.gpu
@pytest.mark.parametrize("n,split", [(9000, False), (30000, True)])
def test_gpu_laplacian_of_rugged_surfaces(n, split):
    """Vertices with more neighbours than the short list holds, on both sides of
    the vertex count from which they have a launch of their own."""
    from water_simulation_amd import mesh as WM

    r = 0.012
    x = np.random.default_rng(n).uniform(0.0, 2.2 * r * n ** (1 / 3), (n, 3)).astype(np.float32)
    opt = dict(radius=r, smooth_pre=0, smooth_sigma=0.8, iso_factor=0.1)
    m = WM.SurfaceMesher()
    m.run(x, smooth_post=0, **opt)
    v, t = m.vertices(), m.triangles()
    assert (len(v) >= 262144) == split
    a, b = np.sort(t[:, [0, 1, 1, 2, 2, 0]].reshape(-1, 2), 1).T
    degree = np.bincount(np.unique(np.stack([a, b], 1), axis=0).ravel(), minlength=len(v))
    assert (degree > 9).sum() > 100 and degree.max() <= 24
    m.run(x, smooth_post=2, **opt)
    want = M.laplacian_smooth(v, t, 2)
    assert np.array_equal(m.triangles(), t)
    assert np.array_equal(m.vertices().view(np.uint32), want.view(np.uint32))
