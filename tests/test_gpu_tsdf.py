"""TSDF fusion and ray casting on the GPU against the oracle, bit for bit:
grids after each fused frame (16-bit depth and the reference's float4 RGBD
input), ray-cast points, normals and shading from fused and unfused poses,
with and without the zero-crossing refinement, grid resampling; at a small
grid and at the reference's own size (256^3 voxels, 320x240). The fused
scene is found on its analytic surfaces."""
import numpy as np
import pytest

from oracle.tsdf import Grid
from recon_amd.tsdf import VoxelGrid, default_params
from _tsdf_scene import normalized_k, pose, render_depth, surface_distance, to_world

pytestmark = pytest.mark.gpu

ORIGIN = (0.0, 0.01, -1600.01)
DIM = (1500.0, 1500.0, 1500.0)
POSES = [pose(), pose(2, -4, (80, -20, 30)), pose(-3, 3, (-60, 40, -50))]
UNFUSED = pose(1, 1, (20, 10, 0))


def _bits_equal(a, b):
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    return a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32))


def _grids(res, W, H):
    print(f"tsdf grid res={res} image={W}x{H}", flush=True)
    g = VoxelGrid(default_params(resolution=res, width=W, height=H))
    o = Grid(res, W, H, ORIGIN, DIM)
    return g, o


@pytest.mark.parametrize("res,W,H", [(64, 160, 120), (128, 160, 120), (256, 320, 240)])
def test_update_and_raycast_match_oracle_bitexact(res, W, H):
    K = normalized_k(W, H)
    g, o = _grids(res, W, H)
    assert _bits_equal(g.read(), o.data)
    for i, T in enumerate(POSES):
        d = np.round(render_depth(T, K, W, H)).astype(np.uint16)
        g.integrate(d, T, K)
        o.update(d.astype(np.float32), T, K)
        assert _bits_equal(g.read(), o.data), f"grid after frame {i}"
        for refine in (True, False):
            for Tr in (T, UNFUSED):
                got = g.raycast(Tr, K, refine)
                exp = o.raycast(Tr, K, refine)
                for name, a, b in zip(("xyz", "normals", "shade"), got, exp):
                    assert _bits_equal(a, b), f"{name} after frame {i}, refine={refine}"
    # the fused scene is where it should be
    xyz, _, _ = g.raycast(UNFUSED, K, True)
    v = xyz[..., 3] > 0
    v[:4] = v[-4:] = False
    v[:, :4] = v[:, -4:] = False
    assert v.mean() > 0.6
    assert np.median(surface_distance(to_world(UNFUSED, xyz))[v]) < 1.0


def test_rgbd_input_matches_oracle_bitexact():
    W, H, res = 160, 120, 64
    K = normalized_k(W, H)
    g, o = _grids(res, W, H)
    mn, mx = 300.0, 7000.0
    for T in POSES[:2]:
        z = render_depth(T, K, W, H).astype(np.float32)
        rgbd = np.zeros((H, W, 4), np.float32)
        rgbd[..., :3] = 0.5
        rgbd[..., 3] = np.where(z > 0, (z - mn) / (mx - mn), 0)[::-1]  # rows bottom-up
        g.set_depth(rgbd)
        g.update(T, K)
        o.update(o.dist_from_rgbd(rgbd), T, K)
        assert _bits_equal(g.read(), o.data)
    assert (g.read()[..., 1] > 0).sum() > 10000


def test_resample_matches_oracle_bitexact():
    W, H, res = 160, 120, 64
    K = normalized_k(W, H)
    src, osrc = _grids(res, W, H)
    for T in POSES:
        d = np.round(render_depth(T, K, W, H)).astype(np.uint16)
        src.integrate(d, T, K)
        osrc.update(d.astype(np.float32), T, K)
    dst, odst = _grids(res, W, H)
    for T in (POSES[1], pose(5, -7, (100, 50, -80))):
        dst.resample_from(src, T)
        odst.resample_from(osrc, T)
        assert _bits_equal(dst.read(), odst.data)
    # the ray cast of a resampled grid (its occupancy is rebuilt by the resampling)
    for refine in (True, False):
        got = dst.raycast(UNFUSED, K, refine)
        exp = odst.raycast(UNFUSED, K, refine)
        for name, a, b in zip(("xyz", "normals", "shade"), got, exp):
            assert _bits_equal(a, b), f"{name} of the resampled grid, refine={refine}"
    # the resampled grid, ray cast from the matching pose, sees the same scene
    T = POSES[1]
    dst.resample_from(src, T)
    a, _, _ = dst.raycast(np.eye(4, dtype=np.float32), K, True)
    b, _, _ = src.raycast(T, K, True)
    v = (a[..., 3] > 0) & (b[..., 3] > 0)
    assert v.mean() > 0.5
    assert np.median(np.abs(a[..., 2] - b[..., 2])[v]) < 2.0


def test_reset_and_argument_errors():
    W, H, res = 96, 72, 32
    K = normalized_k(W, H)
    g, _ = _grids(res, W, H)
    g.integrate(np.full((H, W), 1500, np.uint16), np.eye(4, dtype=np.float32), K)
    assert (g.read()[..., 1] > 0).any()
    g.reset()
    r = g.read()
    assert np.all(r[..., 0] == 1) and np.all(r[..., 1] == 0)
    xyz, _, _ = g.raycast(np.eye(4, dtype=np.float32), K, True)
    assert np.all(xyz == 0)
    other = VoxelGrid(default_params(resolution=64, width=W, height=H))
    with pytest.raises(RuntimeError):
        other.resample_from(g, np.eye(4))
    with pytest.raises(RuntimeError):
        g.resample_from(g, np.eye(4))
    with pytest.raises(ValueError):
        g.set_depth(np.zeros((H + 1, W), np.uint16))


@pytest.mark.parametrize("res,dim,W,H", [(8, (1500.0, 1500.0, 1500.0), 40, 24), (24, (1433.3, 1371.7, 1490.1), 50, 38),
                                         (72, (1433.3, 1371.7, 1490.1), 96, 72), (136, (1500.0, 1500.0, 1500.0), 97, 61),
                                         (264, (1500.0, 1433.3, 1500.0), 64, 48), (520, (1500.0, 1433.3, 1500.0), 64, 48)])
def test_sign_map_and_slice_cull_at_tile_edges_bitexact(res, dim, W, H):
    """Resolutions with partial 16-voxel tiles, one and several skip blocks, both block sizes,
    voxel centres that floats hold and that they round; cameras outside and inside the grid,
    behind the scene and along an axis; surfaces that move, so that signs turn both ways;
    a resampled grid, then fused again."""
    K = normalized_k(W, H)
    print(f"tsdf grid res={res} image={W}x{H} dim={dim}", flush=True)
    params = default_params(resolution=res, width=W, height=H, dim=dim)
    g, o = VoxelGrid(params), Grid(res, W, H, ORIGIN, dim)
    inside = pose(3, 100, (200, 30, -1500))
    views = [pose(), UNFUSED, inside, pose(0, 180, (0, 0, -3600)), pose(90, 0, (10, 1800, -1600))]
    ramp = (600 + 4 * np.arange(W)[None, :] + 3 * np.arange(H)[:, None]).astype(np.uint16)
    d0 = np.round(render_depth(pose(), K, W, H)).astype(np.uint16)
    frames = [(d0, pose()), (np.where(d0 > 400, d0 - 300, 0).astype(np.uint16), pose()), (ramp, inside), (d0, UNFUSED)]

    def check(grid, oracle, what, poses):
        assert _bits_equal(grid.read(), oracle.data), what
        for k, Tr in enumerate(poses):
            for name, a, b in zip(("xyz", "normals", "shade"), grid.raycast(Tr, K, True), oracle.raycast(Tr, K, True)):
                assert _bits_equal(a, b), f"{name}, {what}, view {k}"

    for i, (d, T) in enumerate(frames[:2] if res > 260 else frames):
        g.integrate(d, T, K)
        o.update(d.astype(np.float32), T, K)
        check(g, o, f"frame {i}", views)
    if res > 260:
        return
    dst, odst = VoxelGrid(params), Grid(res, W, H, ORIGIN, dim)
    dst.resample_from(g, POSES[1])
    odst.resample_from(o, POSES[1])
    check(dst, odst, "resampled", views[:3])
    dst.integrate(ramp, inside, K)
    odst.update(ramp.astype(np.float32), inside, K)
    check(dst, odst, "fused after resampling", views[:3])


@pytest.mark.parametrize("res", [8, 40, 264])
def test_resample_at_workgroup_edges(res):
    """Workgroups of 64 x 4 x 4 voxels that end past the grid, and above 256
    voxels their order by XCD with rows of workgroups to spare: grid and ray
    cast (which reads the sign map) bit for bit."""
    W, H = 64, 48
    K = normalized_k(W, H)
    src, osrc = _grids(res, W, H)
    d = np.round(render_depth(POSES[0], K, W, H)).astype(np.uint16)
    src.integrate(d, POSES[0], K)
    osrc.update(d.astype(np.float32), POSES[0], K)
    dst, odst = _grids(res, W, H)
    T = pose(4, -6, (70, 30, -40))
    dst.resample_from(src, T)
    odst.resample_from(osrc, T)
    assert _bits_equal(dst.read(), odst.data)
    for name, a, b in zip(("xyz", "normals", "shade"), dst.raycast(UNFUSED, K, True), odst.raycast(UNFUSED, K, True)):
        assert _bits_equal(a, b), name


def _fused(res, zs, depth, Tcur, K, W, H):
    """One frame fused into the slices zs of a new grid (updateVoxelsKernel in
    float32, every voxel projected): (len(zs), res, res, 2)."""
    f = np.float32
    org, dim = np.array(ORIGIN, f), np.array(DIM, f)
    vs = dim / f(res)
    start, edge = (org - dim) + vs, vs * f(2)
    R, t = np.asarray(Tcur, f)[:3, :3], np.asarray(Tcur, f)[:3, 3]
    i = np.arange(res, dtype=f)
    px, py = (start[0] + i * edge[0])[None, None, :], (start[1] + i * edge[1])[None, :, None]
    pz = (start[2] + np.asarray(zs, f) * edge[2])[:, None, None]
    r = [R[0, k] * px + R[1, k] * py + R[2, k] * pz + -(R[0, k] * t[0] + R[1, k] * t[1] + R[2, k] * t[2]) for k in range(3)]
    dist, vox = np.asarray(depth, f), -r[2]
    with np.errstate(all="ignore"):
        u = (r[0] / r[2] * K[0] + K[2]) * f(W)
        v = (r[1] / r[2] * K[4] + K[5]) * f(H)
        ok = (u >= 1) & (u < W - 2) & (v >= 1) & (v < H - 2)
    u, v = np.where(ok, u, f(1)), np.where(ok, v, f(1))
    ui, vi = u.astype(np.int32), v.astype(np.int32)
    m = [dist[vi + b, ui + a] for b in (0, 1) for a in (0, 1)]
    fu, fv = u - ui.astype(f), v - vi.astype(f)
    d = (1 - fu) * (1 - fv) * m[0] + fu * (1 - fv) * m[1] + (1 - fu) * fv * m[2] + fu * fv * m[3]
    for k in m:
        ok &= (k >= edge[0]) & (np.abs(d - k) <= dim[0] / f(200))
    sdf = -(vox - d) / (dim[0] * f(0.030))
    ok &= sdf >= f(-1.25)
    out = np.empty(ok.shape + (2,), f)
    out[..., 0] = np.where(ok, np.clip(sdf, f(-1), f(1)), f(1))
    out[..., 1] = ok
    return out


def test_slice_cull_at_1024_voxels_an_axis():
    """The largest grid, whose oracle would not fit the host: chosen slices
    against every voxel's own projection in numpy, which equals the oracle on a
    small grid."""
    from recon_amd import lib
    from recon_amd.hip import hip
    W, H, res = 160, 120, 1024
    K = normalized_k(W, H)
    print(f"tsdf grid res={res} image={W}x{H}", flush=True)
    views = [pose(), pose(7, -11, (80, -20, 30)), pose(3, 100, (200, 30, -1500)), pose(0, 180, (0, 0, -3600))]
    for T in views:
        d = np.round(render_depth(T, K, W, H)).astype(np.uint16)
        o = Grid(40, W, H, ORIGIN, DIM)
        o.update(d.astype(np.float32), T, K)
        assert _bits_equal(_fused(40, np.arange(40), d, T, K, W, H), o.data)
    g = VoxelGrid(default_params(resolution=res, width=W, height=H))
    buf, hit = np.empty((res, res, 2), np.float32), 0
    for T in views:
        d = np.round(render_depth(T, K, W, H)).astype(np.uint16)
        g.reset()
        g.integrate(d, T, K)
        g.synchronize()
        for z in (0, 15, 16, 511, 640, 1023):
            assert hip().hipMemcpy(buf.ctypes.data, lib().rt_tsdf_data(g.h) + z * buf.nbytes, buf.nbytes, 2) == 0
            want = _fused(res, [z], d, T, K, W, H)[0]
            hit += int(want[..., 1].sum())
            assert _bits_equal(buf, want), z
    assert hit > 500000
    g.close()


def test_poses_that_are_not_finite_bitexact():
    """Poses and projections that are infinite, huge or not a number: voxels
    whose projection leaves the image stay as they are, and no slice is culled
    that the update would change."""
    W, H, res = 64, 48, 40
    K = normalized_k(W, H)
    d = np.full((H, W), 1500, np.uint16)
    bad = []
    for i, x in ((3, np.nan), (3, np.inf), (11, np.inf), (11, -np.inf), (0, np.nan), (10, np.inf), (7, 1e30), (11, 3e38),
                 (0, 1e38)):
        T = pose(3, 5, (10, 20, 30)).ravel()
        T[i] = x
        bad.append((i, x, T.reshape(4, 4)))
    for i, x, T in bad:
        g, o = _grids(res, W, H)
        g.integrate(d, pose(), K)
        o.update(d.astype(np.float32), pose(), K)
        with np.errstate(all="ignore"):
            g.integrate(d, T, K)
            o.update(d.astype(np.float32), T, K)
        a, b = g.read(), o.data
        assert np.array_equal(a, b, equal_nan=True), (i, x)
