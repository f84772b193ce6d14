"""Parity of the HIP integrate kernel (librecon.so) with the CPU oracle.

Bar: D and W bit-exact with the float32 restatement of cu_tsdf_integrate
(tsdf_volume.cu:144-190 under the build contract), D within 1e-6 absolute of
the float64 decision-matched oracle, update counts equal.
"""
import numpy as np
import pytest

from helpers import assert_bitexact, gpu_run, oracle_run

import oracle_ffi as O
import recon
from recon import scenes

pytestmark = pytest.mark.gpu

F64_TOL = 1e-6  # absolute, metres, for volumes within a few metres of the origin


def _check(w, depth, fused=False, pitch_pad=0, f64=True, f64_tol=F64_TOL):
    cfg = w.config()
    o = oracle_run(cfg, depth, w.poses, f64=f64)
    g = gpu_run(cfg, depth, w.poses, fused=fused, pitch_pad=pitch_pad, count=True)
    assert_bitexact(g["W"], o["W"], "W")
    assert_bitexact(g["D"], o["D"], "D")
    if fused:
        assert int(g["counts"][0]) == int(sum(o["counts"]))
    else:
        assert g["counts"].tolist() == [int(c) for c in o["counts"]]
    if f64:
        err = np.abs(g["D"].astype(np.float64) - o["D64"]).max()
        assert err <= f64_tol, err
        assert np.array_equal(g["W"].astype(np.float64), o["W64"])
    g["vol"].close()
    return o


def test_tiny_exact(cuda):
    w = scenes.tiny()
    o = _check(w, w.render())
    assert sum(o["counts"]) > 0


def test_plain_small_exact(cuda):
    w = scenes.plain_small()
    o = _check(w, w.render())
    assert min(o["counts"]) > 100000


def test_plain_small_fused_equals_per_frame(cuda):
    w = scenes.plain_small()
    _check(w, w.render(), fused=True, f64=False)


@pytest.mark.parametrize("grid", [(37, 29, 23), (66, 8, 9), (4, 4, 4), (1, 1, 1), (130, 5, 7)])
def test_ragged_grids(cuda, grid):
    # gx not a multiple of 4, gy and gz not of the wave-tile's 8 and 2
    w = scenes.tiny(grid=grid, voxel_size=0.6 / max(grid), image=(40, 30), num_frames=4)
    _check(w, w.render())


def test_pitched_depth(cuda):
    w = scenes.tiny(grid=(48, 40, 32), voxel_size=0.02, image=(50, 38), num_frames=3)
    _check(w, w.render(), pitch_pad=13)


def test_weight_cap_and_many_frames(cuda):
    # more frames than max_weight (2): W saturates, D keeps averaging with (W+1)
    w = scenes.tiny(num_frames=20)
    w.poses = np.repeat(w.poses[:2], 10, axis=0)
    o = _check(w, w.render())
    assert o["W"].max() == 2.0


def test_fused_more_than_16_frames(cuda):
    w = scenes.tiny(grid=(32, 32, 32), voxel_size=0.02, num_frames=37)
    _check(w, w.render(), fused=True, f64=False)


def test_invalid_depth_values(cuda):
    w = scenes.tiny(grid=(32, 24, 20), voxel_size=0.03, num_frames=3)
    depth = w.render()
    depth[0, ::3, ::2] = np.nan
    depth[1, 1::4] = np.inf
    depth[2, :, :5] = -1.0
    depth[2, :, 5:9] = 30.0  # beyond max_depth 24
    _check(w, depth, f64=False)


def test_empty_depth_leaves_volume(cuda):
    w = scenes.tiny(num_frames=2)
    depth = np.zeros((2, w.image[1], w.image[0]), np.float32)
    o = _check(w, depth)
    assert sum(o["counts"]) == 0
    assert (o["W"] == 0).all()


def _random_pose_workload(seed, grid=(96, 80, 72), vs=0.01, offset=None, inside=False):
    """Cameras at random positions (inside the volume when `inside`) looking
    at random points of the volume, random-valued depth maps."""
    rng = np.random.default_rng(seed)
    w = scenes.tiny(grid=grid, voxel_size=vs, image=(160, 120), num_frames=6)
    if offset is not None:
        w.offset = offset
    lo = np.array(w.offset)
    hi = lo + np.array(grid) * vs
    poses = []
    for _ in range(w.num_frames):
        if inside:
            c = lo + rng.uniform(0.2, 0.8, 3) * (hi - lo)
        else:
            c = (lo + hi) / 2 + rng.normal(0, 1, 3) * (hi - lo)
        target = lo + rng.uniform(0, 1, 3) * (hi - lo)
        poses.append(scenes.look_at_pose(c, target, up=(0.3, 0.2, 1.0)))
    w.poses = np.array(poses)
    depth = rng.uniform(0.0, 2.0 * np.linalg.norm(hi - lo), (w.num_frames, 120, 160)).astype(np.float32)
    depth[rng.random(depth.shape) < 0.3] = 0.0
    # patches of constant depth exercise the block bounds
    depth[:, 20:60, 40:100] = rng.uniform(0.05, 1.0)
    return w, depth


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_cull_random_poses_outside(cuda, seed):
    w, depth = _random_pose_workload(seed)
    _check(w, depth)


@pytest.mark.parametrize("seed", [4, 5])
def test_cull_camera_inside_volume(cuda, seed):
    w, depth = _random_pose_workload(seed, inside=True)
    _check(w, depth)


def test_cull_far_from_origin(cuda):
    # 70 m from the origin a float32 ulp is 7.6e-6 m, so the float64 bound
    # scales with the coordinates: 4 ulp of the largest coordinate
    w, depth = _random_pose_workload(6, vs=0.02, offset=(50.0, -70.0, 30.0), inside=True)
    _check(w, depth, f64_tol=4 * 2.0 ** -23 * 72.0)
    w, depth = _random_pose_workload(7, vs=0.02, offset=(50.0, -70.0, 30.0))
    _check(w, depth, fused=True, f64=False)


def test_cull_fused_random(cuda):
    w, depth = _random_pose_workload(8, inside=True)
    w.poses = np.concatenate([w.poses] * 4)
    depth = np.concatenate([depth] * 4)
    _check(w, depth, fused=True, f64=False)


@pytest.mark.parametrize("gz", [256, 258])
def test_cull_segment_limits(cuda, gz):
    # 2048 x 1024 x gz voxels (4 GB of D and W): 64 x 128 x gz/2 wave-tiles of
    # 32 x 8 x 2.  gz = 256 gives 4096 x 256 tiles, the most cull segments of
    # 256 tiles; gz = 258 gives more, so segments of 512 tiles.  Per-frame and
    # fused calls, bit-exact, update counts equal.
    w = scenes.tiny(grid=(2048, 1024, gz), voxel_size=0.001, image=(320, 240), num_frames=2)
    cfg = w.config()
    depth = w.render()
    o = oracle_run(cfg, depth, w.poses)
    assert min(o["counts"]) > 100_000_000
    for fused in (False, True):
        g = gpu_run(cfg, depth, w.poses, fused=fused, count=True)
        assert_bitexact(g["W"], o["W"], "W")
        assert_bitexact(g["D"], o["D"], "D")
        if fused:
            assert int(g["counts"][0]) == int(sum(o["counts"]))
        else:
            assert g["counts"].tolist() == [int(c) for c in o["counts"]]
        g["vol"].close()
        del g


def test_touch_counter_is_union_per_sweep(cuda):
    """recon_tsdf_set_touch_counter: per-frame calls count each updated voxel
    once (= the update count); a fused call counts, per sweep of 16 frames,
    the voxels that any of its frames updates (the oracle's masks OR-ed)."""
    import recon
    import oracle_ffi as O

    w = scenes.tiny(grid=(40, 36, 28), voxel_size=0.025, image=(64, 48), num_frames=21)
    depth = w.render()
    cfg = w.config()
    ov = O.volume_from_config(cfg)
    D, W = O.init(ov)
    masks = []
    for f in range(w.num_frames):
        n, m = O.integrate_f32(ov, D, W, depth[f], w.poses[f], mask=True)
        assert int((m != 0).sum()) == n
        masks.append(m != 0)
    dev = cuda.from_numpy(depth).cuda()
    vol = recon.TSDFVolume(cfg)
    t = cuda.zeros(w.num_frames, dtype=cuda.int64, device="cuda")
    for f in range(w.num_frames):
        vol.set_touch_counter(t[f:f + 1])
        vol.integrate(dev[f], w.poses[f])
    vol.set_touch_counter(None)
    vol.reset()
    u = cuda.zeros(1, dtype=cuda.int64, device="cuda")
    vol.set_touch_counter(u)
    vol.integrate_frames(dev, w.poses)
    vol.set_touch_counter(None)
    cuda.cuda.synchronize()
    assert t.cpu().numpy().tolist() == [int(m.sum()) for m in masks]
    union = sum(int(np.logical_or.reduce(masks[a:a + 16]).sum()) for a in range(0, w.num_frames, 16))
    assert int(u.item()) == union > 0
    Dg, Wg = vol.download()
    assert_bitexact(Wg, W, "fused W")
    assert_bitexact(Dg, D, "fused D")
    vol.close()


@pytest.mark.parametrize("weight_type", [0, 1])
@pytest.mark.parametrize("grid", [(1, 1, 1), (31, 7, 1), (33, 9, 3), (65, 17, 9), (37, 64, 50),
                                  (256, 256, 256), (256, 256, 257)])
def test_direct_and_list_kernels_agree(cuda, grid, weight_type):
    """Small volumes take one launch without cull or list; a counted call
    takes the list kernel at any size: equal bits, on both sides of the size
    rule (32768 wave-tiles of 32 x 8 x 2) and at ragged edges."""
    w = scenes.tiny(grid=grid, voxel_size=0.8 / max(grid), image=(96, 72), num_frames=3)
    depth = cuda.from_numpy(w.render()).cuda()
    cfg = w.config()
    cfg.weight_type = weight_type
    counter = cuda.zeros(1, dtype=cuda.int64, device="cuda")
    got = []
    for counted in (False, True):
        v = recon.TSDFVolume(cfg)
        v.set_update_counter(counter if counted else None)
        for f in range(w.num_frames):
            v.integrate(depth[f], w.poses[f])
        cuda.cuda.synchronize()
        got.append(v.download())
        v.close()
    assert_bitexact(got[0][0], got[1][0], "D")
    assert_bitexact(got[0][1], got[1][1], "W")


# Poses turned by 4e-36 about an axis of the image: the camera z of a layer
# through the camera centre is 4e-36 x or y, a normal number, and x * f / z
# overflows.  Such a voxel projects to no pixel.  The grids have a wave-tile
# (32 x 8 x 2) across the optical axis, which the frustum test keeps.
GRAZING_POSES = np.array([[1, 0, -2e-36, 0, 0, 0, 0], [1, 2e-36, 0, 0, 0, 0, 0],
                          [1, 0, 2e-36, 0, 0, 0, 0]], np.float64)


def _grazing_workload(grid):
    w = scenes.tiny(grid=grid, voxel_size=1 / 64, image=(640, 480), num_frames=3)
    # voxel centres of layer gz / 2 at z = 0 exactly
    w.offset = (-grid[0] / 128, -grid[1] / 128, -(grid[2] // 2 + 0.5) / 64)
    w.intrinsics = (2000.0, 2000.0, 319.5, 239.5)
    w.poses = GRAZING_POSES
    return w, np.full((3, 480, 640), 1.0, np.float32)


@pytest.mark.parametrize("path", ["single", "counted", "fused", "batch"])
@pytest.mark.parametrize("grid", [(96, 40, 32), (63, 40, 32), (288, 248, 257), (287, 248, 257)])
def test_layer_through_the_camera_centre(cuda, grid, path):
    w, depth = _grazing_workload(grid)
    cfg = w.config()
    o = oracle_run(cfg, depth, w.poses)
    assert (o["W"] > 0).any() and (o["W"][grid[2] // 2] == 0).all()
    if path == "batch":
        b = recon.Batch([(cfg, cuda.from_numpy(depth).cuda(), w.poses)])
        b.run()
        cuda.cuda.synchronize()
        D, W = b.download(0)
        b.close()
    else:
        g = gpu_run(cfg, depth, w.poses, fused=path == "fused", count=path == "counted")
        D, W = g["D"], g["W"]
        g["vol"].close()
    assert_bitexact(W, o["W"], "W")
    assert_bitexact(D, o["D"], "D")


def _extreme_state(shape, seed):
    """D and W as a caller may upload them: sentinels, overflowing and
    vanishing products, whole and fractional weights; weights whose reciprocal
    is not normal in half of the layers only."""
    rng = np.random.default_rng(seed)
    d = np.array([0.0, 0.02, -0.03, np.inf, -np.inf, np.nan, 1e-40, -3e-33, 1e-20, 3e38, 1e30], np.float32)
    k = np.array([0.0, 0.5, 1.0, 7.25, 127.0, 255.0, 300.0, 1e-30, 1e30, 3e38], np.float32)
    W = rng.choice(k[:-2], shape)
    W[2::4] = rng.choice(k, W[2::4].shape)
    W[3::4] = rng.choice(k, W[3::4].shape)
    return rng.choice(d, shape), W


def _assert_same_values(a, b, what):
    # any NaN equals any NaN: its sign and payload are not part of the contract
    assert np.array_equal(np.isnan(a), np.isnan(b)), what
    assert_bitexact(np.where(np.isnan(a), np.float32(0), a), np.where(np.isnan(b), np.float32(0), b), what)


@pytest.mark.parametrize("path", ["single", "counted", "fused", "diff"])
@pytest.mark.parametrize("grid,weight_type", [((64, 40, 32), 0), ((63, 40, 32), 0), ((64, 40, 32), 1),
                                              ((256, 256, 257), 0), ((257, 256, 257), 1)])
def test_uploaded_extremes(cuda, grid, weight_type, path):
    """One update of a volume whose D and W came from outside: the quotient
    of the running average is the division's also where it overflows, is not a
    number or is close to the denormals (a layer at the observed depth, where
    the update adds exactly 0)."""
    if path == "diff" and weight_type:
        pytest.skip("the differentiable integrate weighs every observation 1")
    w = scenes.tiny(grid=grid, voxel_size=1 / 64, image=(160, 120), num_frames=2)
    w.intrinsics = (140.0, 140.0, 79.5, 59.5)
    w.max_weight = 1e30
    w.truncation = 0.0625
    w.poses = np.array([[1, 0, 0, 0, 0, 0, 3], [1, 0, 0, 0, 0.5, 0, 3]], np.float64)
    depth = np.full((2, 120, 160), 3.0 + 0.5 / 64 + (grid[2] % 2) * 0.5 / 64, np.float32)
    depth[:, ::7, ::5] = 0.0
    frames = 2 if path in ("fused", "diff") else 1
    cfg = w.config()
    cfg.weight_type = weight_type
    vol = O.volume_from_config(cfg)
    D, W = O.init(vol)
    D[...], W[...] = _extreme_state(D.shape, sum(grid))
    v = recon.TSDFVolume(cfg)
    v.upload(D, W)
    dev = cuda.from_numpy(depth).cuda()
    counter = cuda.zeros(1, dtype=cuda.int64, device="cuda")
    v.set_update_counter(counter if path == "counted" else None)
    before = W.copy()
    if path == "diff":
        rt = recon.pose_to_matrix(w.poses).astype(np.float32)
        v.diff_integrate(dev, cuda.from_numpy(rt).cuda())
        O.lib().oracle_diff_forward_f32(O.C.byref(vol), O._p(D), O._p(W), O._p(depth), 120, 160,
                                        O._p(np.ascontiguousarray(rt)), 2, 0)
    else:
        if path == "fused":
            v.integrate_frames(dev, w.poses)
        else:
            v.integrate(dev[0], w.poses[0])
        for f in range(frames):
            O.integrate_f32(vol, D, W, depth[f], w.poses[f])
    cuda.cuda.synchronize()
    Dg, Wg = v.download()
    v.close()
    assert (W != before).sum() > 100
    _assert_same_values(Wg, W, "W")
    _assert_same_values(Dg, D, "D")


@pytest.mark.parametrize("weight_type", [0, 1])
@pytest.mark.parametrize("grid", [(256, 256, 257), (257, 256, 257)])
def test_list_kernels_equal_oracle(cuda, grid, weight_type):
    """One frame a call into a volume just above 32768 wave-tiles, uncounted:
    the list kernel with lanes of four voxels (gx % 4 == 0) and of a row."""
    w = scenes.tiny(grid=grid, voxel_size=0.8 / max(grid), image=(96, 72), num_frames=2)
    cfg = w.config()
    cfg.weight_type = weight_type
    depth = w.render()
    o = oracle_run(cfg, depth, w.poses)
    assert min(o["counts"]) > 100000
    g = gpu_run(cfg, depth, w.poses)
    assert_bitexact(g["W"], o["W"], "W")
    assert_bitexact(g["D"], o["D"], "D")
    g["vol"].close()


@pytest.mark.parametrize("path", ["single", "counted", "fused", "batch", "diff"])
def test_row_stride_beyond_24_bits(cuda, path):
    """Rows 2^22 floats apart: their byte offsets do not fit the 24-bit products
    of the short forms, so the whole frame takes the divisions and 64-bit
    addresses."""
    w = scenes.tiny(grid=(61, 37, 29), voxel_size=0.02, image=(64, 12), num_frames=2)
    depth = w.render()
    o = oracle_run(w.config(), depth, w.poses)
    assert min(o["counts"]) > 1000
    if path in ("batch", "diff"):
        buf = cuda.zeros((2, 12, 1 << 22), dtype=cuda.float32, device="cuda")
        buf[:, :, :64] = cuda.from_numpy(depth).cuda()
    if path == "diff":
        rt = recon.pose_to_matrix(w.poses).astype(np.float32)
        o["D"], o["W"] = O.diff_forward_f32(o["vol"], depth, rt)
        v = recon.TSDFVolume(w.config())
        v.diff_integrate(buf[:, :, :64], cuda.from_numpy(rt).cuda())
        cuda.cuda.synchronize()
        D, W = v.download()
        v.close()
    elif path == "batch":
        b = recon.Batch([(w.config(), buf[:, :, :64], w.poses)])
        b.run()
        cuda.cuda.synchronize()
        D, W = b.download(0)
        b.close()
    else:
        g = gpu_run(w.config(), depth, w.poses, fused=path == "fused", count=path == "counted",
                    pitch_pad=(1 << 22) - 64)
        D, W = g["D"], g["W"]
        g["vol"].close()
    assert_bitexact(W, o["W"], "W")
    assert_bitexact(D, o["D"], "D")
