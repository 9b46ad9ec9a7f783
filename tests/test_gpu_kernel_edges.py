"""Edges of the kernels' tiles and dispatch rules, against the oracle."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import announce, small_sequence

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kf():
    import kfusion
    kfusion.init()
    return kfusion


def same(got, ref, what):
    """The same bits, any NaN for a NaN (its sign and payload are the platform's)."""
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan, err_msg=what)
    np.testing.assert_array_equal(np.where(nan, 0, got.view(np.uint32)), np.where(nan, 0, ref.view(np.uint32)),
                                  err_msg=what)


# (w, h, levels): one pixel, under and over the 16-pixel tile and the 32-pixel region, odd sizes, and
# sizes whose last region holds one coarse pixel
@pytest.mark.parametrize("w,h,levels", [(1, 1, 1), (15, 17, 1), (33, 31, 1), (2, 2, 2), (34, 62, 2), (66, 18, 2),
                                        (4, 4, 3), (28, 32, 3), (36, 68, 3), (132, 100, 3)])
@pytest.mark.parametrize("mirrored", [0, 1])
@pytest.mark.parametrize("normals", [0, 1])
def test_preprocess_edges_bit_exact(kf, oracle32, w, h, levels, mirrored, normals):
    announce(f"kf_preprocess {w}x{h}, {levels} levels, mirrored {mirrored}, normals {normals}")
    rng = np.random.default_rng(100 * w + h)
    raw_h = (1500 + 400 * rng.random((h, w))).astype(np.uint16)
    raw_h[rng.random((h, w)) < 0.05] = 0       # holes
    raw_h[rng.random((h, w)) < 0.02] = 65535   # +inf codes
    raw = kf.DeviceArray.from_host(raw_h)
    dm = kf.GridMap(w, h)
    dp = [kf.GridMap(w >> l, h >> l) for l in range(levels)]
    vp = [kf.GridMap(w >> l, h >> l, 4) for l in range(levels)]
    npm = [kf.GridMap(w >> l, h >> l, 4) for l in range(levels)]
    Ks = [oracle32.intrinsics(525.0, 525.0, w / 2 - 0.5, h / 2 - 0.5, l) for l in range(3)]
    kinv = np.ascontiguousarray(np.stack([k[1] for k in Ks]))
    arr = lambda maps: (C.c_void_p * levels)(*[m.ptr.value for m in maps])  # noqa: E731
    kf.check(kf.lib().kf_preprocess(raw.ptr, w, h, 1e-3, mirrored, levels, kinv.ctypes.data_as(C.c_void_p), dm.ptr,
                                    arr(dp), arr(vp), arr(npm) if normals else None, None, None), "kf_preprocess")
    kf.check(kf.lib().kf_device_synchronize())
    ref = oracle32.convert_to_depth_meters(raw_h, 1e-3, bool(mirrored))
    same(dm.download(), ref, "metres")
    d = oracle32.apply_bilateral_filter(ref)
    for l in range(levels):
        if l:
            d = oracle32.down_sample(d)
        v = oracle32.create_vertex_map(d, Ks[l][1])
        same(dp[l].download(), d, f"depth L{l}")
        same(vp[l].download(), v, f"vertex L{l}")
        if normals:
            same(npm[l].download(), oracle32.create_normal_map(v), f"normal L{l}")


# Sparse volumes: free space with scattered voxels on either side of the two values that matter to a
# march (0.991 on large steps, 0 on small ones), so rays run through boxes of free bricks of every size
# and end, shorten their step or graze at their faces.  n = 8: one brick; 40 and 136: rows that are no
# multiple of the 8-brick tiles; 528: rows of more than 64 bricks.  4 m and n a power of two take the
# march's exact texel coordinates, the others its divisions.
@pytest.mark.parametrize("n,L,mue", [(8, 2.0, 0.05), (40, 2.5, 0.05), (64, 4.0, 0.1), (128, 4.0, 0.02),
                                     (136, 3.0, 0.03), (528, 5.0, 0.03)])
@pytest.mark.parametrize("density", [2e-5, 1e-3])
def test_raycast_sparse_volume_bit_exact(kf, oracle32, n, L, mue, density):
    w, h = 64, 48
    rng = np.random.default_rng(n)
    F = np.full(n ** 3, 1.0, np.float32)
    F[rng.random(n ** 3, np.float32) < 0.3 * min(1.0, 64 / n)] = 2.0  # unobserved
    hits = rng.integers(0, n ** 3, max(4, int(density * n ** 3)))
    F[hits] = rng.choice(np.array([0.992, 0.9909, 0.98, 0.3, 0.0, -0.01, -0.6, -1.0], np.float32), hits.size)
    slab = F.reshape(n, n, n)
    slab[-1 - n // 5:, :, :] *= -1.0  # something to end at
    grid = kf.VoxelGrid(L, n, mue=mue)
    grid.upload(F, np.ones(n ** 3, np.float32))
    sensor = kf.Sensor(60.0, 60.0, w / 2 - 0.5, h / 2 - 0.5)
    vm, nm = kf.GridMap(w, h, 4), kf.GridMap(w, h, 4)
    init = np.zeros((h, w, 4), np.float32)
    init[..., 3] = -2
    for k, (eye, turn) in enumerate([((0.1 * L, -0.05 * L, -0.45 * L), 0.0), ((-0.6 * L, 0.0, 0.1 * L), 1.2),
                                     ((0.0, 0.0, 0.0), 0.7)]):
        pose = np.eye(4, dtype=np.float64)
        pose[0, 0] = pose[2, 2] = np.cos(turn)
        pose[0, 2], pose[2, 0] = np.sin(turn), -np.sin(turn)
        pose[:3, 3] = eye
        sensor.set_pose(pose.T.reshape(-1).astype(np.float32))
        announce(f"raycast sparse n {n} L {L} mue {mue} density {density} pose {k}")
        vm.upload(init)
        nm.upload(init)
        kf.kernel.raycast(grid, sensor, vm, nm, 0)
        rv, rn = oracle32.raycast(F, n, L, mue, sensor.get_pose(), sensor.get_inverse_intr(0), w, h, init.copy(),
                                  init.copy())
        same(vm.download(), rv, f"vertex pose {k}")
        same(nm.download(), rn, f"normal pose {k}")


# (w, h): a map with one full stencil, one workgroup partly and just filled, one pixel over it, 64 and 65
# partial rows (one and two per lane of the sum), and more rows than one round of loads takes (320)
@pytest.mark.parametrize("w,h", [(2, 2), (33, 31), (32, 32), (41, 25), (256, 256), (260, 256), (1300, 260)])
@pytest.mark.parametrize("comp", [False, True])
def test_icp_reduce_edges(kf, w, h, comp):
    """The fused reduction against the FP64 sums of the rows kf_construct_icp_residuals writes.  Every
    product is fused into a lane's sum of at most 4 rows (4 roundings of 2^-24 of the sum of the
    products' magnitudes); the plain form then rounds at each of 6 lane steps, 3 waves, ceil(rows / 64)
    partial rows and 6 lane steps more, the compensated form adds in FP64."""
    announce(f"kf_icp_reduce {w}x{h} compensated {comp}")
    rng = np.random.default_rng(7 * w + h)
    f = 1.2 * w
    u, v = np.meshgrid(np.arange(w) + 0.5, np.arange(h) + 0.5)
    z = 2.0 + 0.1 / w * rng.random((h, w))
    V = np.stack([(u - w / 2) / f * z, (v - h / 2) / f * z, z, np.full((h, w), -1.0)], -1).astype(np.float32)
    holes = rng.random((h, w)) < 0.03
    holes[:2, :2] = False  # at least one pixel keeps its row
    V[holes] = (0, 0, 0, -2)
    TV = V.copy()
    TV[..., :3] += (0.02 * rng.random((h, w, 3)) - 0.01).astype(np.float32)
    N = np.concatenate([0.2 * rng.random((h, w, 2)) - 0.1, np.ones((h, w, 1))], -1)
    TN = np.concatenate([N / np.linalg.norm(N, axis=-1, keepdims=True), np.full((h, w, 1), -1.0)], -1)
    TN = TN.astype(np.float32)
    maps = []
    for m in (V, TV, TN):
        g = kf.GridMap(w, h, 4)
        g.upload(m)
        maps.append(g)
    R, t = np.eye(3, dtype=np.float32).reshape(9), np.zeros(3, np.float32)
    K = np.array([f, 0, 0, 0, f, 0, w / 2, h / 2, 1], np.float32)
    th = float(np.deg2rad(60.0))
    A, b = kf.DeviceArray((h * w, 6)), kf.DeviceArray((h * w,))
    kf.kernel.construct_icp_residuals(*maps, R, t, R, t, K, 0.1, th, A, b)
    rows = np.concatenate([A.download(), b.download()[:, None]], 1).astype(np.float64)
    hits = int(np.any(rows[:, :6] != 0, axis=1).sum())
    assert hits > 0
    p, q = [np.concatenate([x, y]) for x, y in zip(np.triu_indices(6), (np.arange(6), np.full(6, 6)))]
    prod = rows[:, p] * rows[:, q]
    sums, inliers = kf.kernel.icp_reduce(*maps, R, t, R, t, K, 0.1, th, compensated=comp)
    assert inliers == hits
    blocks = -(-w * h // 1024)
    roundings = 4 if comp else 4 + 6 + 3 + -(-blocks // 64) + 6
    bound = 1.01 * roundings * 2.0 ** -24 * np.abs(prod).sum(0)
    assert (np.abs(sums - prod.sum(0)) <= bound).all()


@pytest.mark.parametrize("w,h", [(64, 48), (2, 300), (300, 2)])
def test_projection_at_pixel_borders_bit_exact(kf, oracle32, w, h):
    """A pixel's target is the floor of its projection, taken from approximate quotients except near
    an integer: projections on the pixel borders and within 3 ulps of them, off the map, behind the
    camera and at depths beyond the approximation's range, every row against the oracle's.  The
    thresholds accept any target, so a wrong one shows."""
    announce(f"projection at pixel borders {w}x{h}")
    rng = np.random.default_rng(w)
    z = (0.4 + 5.6 * rng.random((h, w))).astype(np.float32)
    z[rng.random((h, w)) < 0.1] *= -1
    scale = rng.choice([1.0, 1e-33, 1e33], size=(h, w), p=[0.9, 0.05, 0.05]).astype(np.float32)
    z = z * scale
    k, l = rng.integers(-2, w + 3, (h, w)), rng.integers(-2, h + 3, (h, w))
    ulp = lambda: 1 + rng.integers(-3, 4, (h, w)).astype(np.float32) * np.float32(2.0 ** -23)  # noqa: E731
    V = np.stack([k.astype(np.float32) * z * ulp(), l.astype(np.float32) * z * ulp(), z, np.full((h, w), -1.0)], -1)
    V = V.astype(np.float32)
    TV = np.concatenate([rng.standard_normal((h, w, 3)), np.full((h, w, 1), -1.0)], -1).astype(np.float32)
    N = rng.standard_normal((h, w, 3))
    TN = np.concatenate([N / np.linalg.norm(N, axis=-1, keepdims=True), np.full((h, w, 1), -1.0)], -1)
    TN = TN.astype(np.float32)
    maps = []
    for m in (V, TV, TN):
        g = kf.GridMap(w, h, 4)
        g.upload(m)
        maps.append(g)
    R, t = np.eye(3, dtype=np.float32).reshape(9), np.zeros(3, np.float32)
    K = np.eye(3, dtype=np.float32).reshape(9)
    A, b = kf.DeviceArray((h * w, 6)), kf.DeviceArray((h * w,))
    kf.kernel.construct_icp_residuals(*maps, R, t, R, t, K, 1e18, float(np.pi), A, b)
    Ar, br = oracle32.construct_icp_residuals(V, TV, TN, R, t, R, t, K, 1e18, float(np.pi))
    assert np.count_nonzero(np.any(Ar != 0, axis=1)) > 0.1 * w * h
    same(A.download(), Ar, "A")
    same(b.download(), br, "b")
    # the fused reduction takes its targets by 32-bit offsets: the same rows are counted
    _, inliers = kf.kernel.icp_reduce(*maps, R, t, R, t, K, 1e18, float(np.pi))
    assert inliers == np.count_nonzero(np.any(Ar != 0, axis=1) | (br != 0))


# one chunk, one thread with two chunks and a remainder, two threads, four threads with a remainder
@pytest.mark.parametrize("n", [8, 72, 104, 136])
@pytest.mark.parametrize("fmt", [0, 1])
def test_volume_to_host_and_back(kf, tmp_path, n, fmt):
    """Every voxel arrives where it left: random values uploaded, downloaded, saved, loaded into another
    volume and drawn alike (the precision form's values are representable: codes and whole counts)."""
    announce(f"volume transfer {n}^3 format {fmt}")
    rng = np.random.default_rng(n)
    if fmt == 0:
        F, W = rng.standard_normal((2, n, n, n)).astype(np.float32)
    else:
        F = rng.integers(-32767, 32768, (n, n, n)).astype(np.float32) * (np.float32(1) / np.float32(32767))
        W = rng.integers(0, 129, (n, n, n)).astype(np.float32)
    fw = np.ascontiguousarray(np.stack([F, W], -1))
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    a, b = [kf.VoxelGrid(3.0, n, mue=0.03, voxel_format=fmt) for _ in range(2)]
    kf.check(kf.lib().kf_volume_upload(a.h, p(fw)))
    back = np.zeros_like(fw)
    kf.check(kf.lib().kf_volume_download(a.h, p(back)))
    np.testing.assert_array_equal(back.view(np.uint32), fw.view(np.uint32))
    path = str(tmp_path / "v.bin").encode()
    kf.check(kf.lib().kf_volume_save(a.h, path))
    np.testing.assert_array_equal(np.fromfile(path.decode(), np.uint32), fw.view(np.uint32).reshape(-1))
    kf.check(kf.lib().kf_volume_load(b.h, path))
    kf.check(kf.lib().kf_volume_download(b.h, p(back)))
    np.testing.assert_array_equal(back.view(np.uint32), fw.view(np.uint32))
    with open(path.decode(), "r+b") as f:
        f.truncate(fw.nbytes - 8)
    assert kf.lib().kf_volume_load(b.h, path) == kf.KF_ERR_IO
    a.close()
    b.close()


@pytest.mark.parametrize("n,w,h", [(200, 320, 240), (96, 200, 148)])
def test_free_bricks_bit_exact(kf, oracle32, n, w, h):
    """Bricks in free space are updated without projecting their voxels: a wall seen over an object
    that comes and goes, with holes, infinite and NaN depths, into a volume that holds random codes and
    counts (127 and 128 among them) in places, against the oracle voxel by voxel."""
    announce(f"free bricks n {n} {w}x{h}")
    L, mue = 2.0, 0.03
    rng = np.random.default_rng(n)
    Fq, Wq = oracle32.new_volume_q(n)
    some = rng.random((n // 8,) * 3) < 0.3
    some = np.repeat(np.repeat(np.repeat(some, 8, 0), 8, 1), 8, 2).reshape(-1)
    Fq[some] = rng.choice(np.array([32767, 32767, 32767, 20000, -500], np.int16), int(some.sum()))
    Wq[some] = rng.choice(np.array([1, 5, 127, 128], np.uint8), int(some.sum()))
    inv = np.float32(1) / np.float32(32767)
    F = np.where(Fq == -32768, np.float32(2), Fq.astype(np.float32) * inv)
    fw = np.ascontiguousarray(np.stack([F, Wq.astype(np.float32)], -1))
    grid = kf.VoxelGrid(L, n, mue=mue, voxel_format=kf.KF_VOXEL_SNORM16_U8)
    kf.check(kf.lib().kf_volume_upload(grid.h, fw.ctypes.data_as(C.c_void_p)))
    sensor = kf.Sensor(0.82 * w, 0.82 * w, w / 2 - 0.5, h / 2 - 0.5)
    dm = kf.GridMap(w, h)
    touched = 0
    for f in range(4):
        d = (1.9 + 0.1 * np.sin(np.arange(w) / 17.0)[None, :] + 0.05 * rng.random((h, w))).astype(np.float32)
        if f % 2:
            d[h // 4:h // 2, w // 4:w // 2] = 0.9
        d[rng.random((h, w)) < 2e-4] = 0.0
        d[3 * h // 4, : w // 3] = np.inf
        d[h - 9, w // 2] = np.nan
        pose = np.eye(4, dtype=np.float32)
        pose[3, :3] = (0.02 * f, 0.01 * f, -1.35)  # column-major
        sensor.set_pose(pose.reshape(-1))
        dm.upload(d)
        kf.kernel.fuse(dm, grid, sensor)
        touched += oracle32.fuse_q(Fq, Wq, n, L, mue, d, sensor.get_inverse_pose(), sensor.get_intr(0))
    Fg, Wg = grid.download()
    np.testing.assert_array_equal(Wg.reshape(-1), Wq.astype(np.float32))
    np.testing.assert_array_equal(Fg.reshape(-1), np.where(Fq == -32768, np.float32(2), Fq.astype(np.float32) * inv))
    assert grid.touched_total() == touched > 0.1 * n ** 3


# either side of the largest frame whose normals are formed by 16x16 regions (600000 pixels), and maps
# without normals, formed in one pass
@pytest.mark.parametrize("w,h,normals", [(960, 624, 1), (964, 624, 1), (644, 484, 0)])
def test_preprocess_one_or_two_passes(kf, oracle32, w, h, normals):
    test_preprocess_edges_bit_exact(kf, oracle32, w, h, 3, 1, normals)


def test_solve_from_several_threads(kf):
    """One call at a time has the fixed working memory and the pinned result, the others allocate: every
    thread gets its own system's solution, bit for bit the one it gets alone, and its own status."""
    import threading

    announce("solve from four threads")
    rng = np.random.default_rng(3)
    lib, sets = kf.lib(), []
    for n in (7, 1000, 5000, 70000):
        A, b = rng.standard_normal((n, 6)).astype(np.float32), rng.standard_normal(n).astype(np.float32)
        sets.append([kf.DeviceArray.from_host(A), kf.DeviceArray.from_host(b), n])
    sets[1][0] = kf.DeviceArray.from_host(np.zeros((1000, 6), np.float32))  # not positive definite

    def solve(s):
        x = np.full(6, 9.0, np.float32)
        return lib.kf_solve_normal_equations(s[0].ptr, s[1].ptr, s[2], x.ctypes.data_as(C.c_void_p), None, None), x

    alone = [solve(s) for s in sets]
    assert [r[0] for r in alone] == [0, kf.KF_ERR_NOT_PD, 0, 0] and (alone[1][1] == 0).all()
    got = [[] for _ in sets]
    threads = [threading.Thread(target=lambda k=k: got[k].extend(solve(sets[k]) for _ in range(50))) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(4):
        assert len(got[k]) == 50
        for rc, x in got[k]:
            assert rc == alone[k][0]
            np.testing.assert_array_equal(x, alone[k][1])
