"""Mapping through every route that fuses or draws a volume (single calls, the frame loop, batch ticks):
frames that are not fused, uploaded states, volumes of more than 64 bricks a side."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import announce, decode_q, small_sequence

pytestmark = pytest.mark.gpu

TH = float(np.deg2rad(20.0))


@pytest.fixture(scope="module")
def kf():
    import kfusion
    kfusion.init()
    return kfusion


def make_pipeline(kf, seq, n, fmt, iters=(4, 3, 2), **kw):
    w, h = seq.width, seq.height
    return kf.Pipeline(w, h, seq.fx, seq.fy, seq.cx, seq.cy, 1e-3, n, seq.L, 0.03, voxel_format=fmt,
                       initial_pose=seq.pose(0), icp=kf.IcpConfig(iters, w, h, 0.1, TH, compensated=True), **kw)


def make_batch(kf, seq, n, fmt, iters=(4, 3, 2), sessions=1, **kw):
    w, h = seq.width, seq.height
    b = kf.Batch(sessions, icp=kf.IcpConfig(iters, w, h, 0.1, TH, compensated=True), **kw)
    cfg = kf.SessionConfig(w, h, seq.fx, seq.fy, seq.cx, seq.cy, 1e-3, n, seq.L, 0.03, fmt, seq.pose(0))
    return b, [b.add(cfg) for _ in range(sessions)]


def upload(kf, handle, F, W):
    fw = np.ascontiguousarray(np.stack([F, W.astype(np.float32)], -1))
    kf.check(kf.lib().kf_volume_upload(handle, fw.ctypes.data_as(C.c_void_p)))


def batch_volume(kf, b, sid):
    v = C.c_void_p()
    kf.check(kf.lib().kf_batch_volume(b.h, sid, C.byref(v)))
    return v


# blank frames between the others: none, one, two in a row, two apart
@pytest.mark.parametrize("blanks", [(), (2,), (2, 3), (2, 4)])
@pytest.mark.parametrize("fmt", [0, 1])
def test_frames_that_are_not_fused(kf, blanks, fmt):
    """A blank frame's ICP fails: it is reported and leaves the model as it is, and the frames after it
    are fused once each, as if it had not come (pose, every voxel, every predicted map and the count of
    fused voxels), in the frame loop and in a batch."""
    seq = small_sequence(seed=11, n_frames=4, w=160, h=120, L=3.0)
    raws = seq.frames(0, 4)
    n = 64
    frames, f = [], 0
    while f < len(raws) or len(frames) in blanks:
        if len(frames) in blanks:
            frames.append(np.zeros_like(raws[0]))
        else:
            frames.append(raws[f])
            f += 1
    dev = kf.DeviceArray.from_host(np.stack(frames))
    plain = kf.DeviceArray.from_host(raws)
    ref = make_pipeline(kf, seq, n, fmt)
    for k in range(len(raws)):
        ref.frame(plain.ptr.value + k * raws[0].nbytes)
    assert ref.sync() == 0
    gp = make_pipeline(kf, seq, n, fmt)
    b, (sid,) = make_batch(kf, seq, n, fmt)
    for k in range(len(frames)):
        announce(f"frame {k} of {len(frames)}, blank {blanks}, format {fmt}")
        gp.frame(dev.ptr.value + k * raws[0].nbytes)
        assert (gp.sync() == kf.KF_ERR_NOT_PD) == (k in blanks)
        b.tick([sid], [dev.ptr.value + k * raws[0].nbytes])
        assert (b.status(sid) == kf.KF_ERR_NOT_PD) == (k in blanks)
    want = ref.volume_download()
    for what, pose, vol, maps, touched in [
            ("loop", gp.pose(), gp.volume_download(), gp.map, gp.touched_total()),
            ("batch", b.pose(sid), b.volume_download(sid), lambda m, l: b.map(sid, m, l), b.touched_total())]:
        np.testing.assert_array_equal(pose, ref.pose(), err_msg=what)
        assert touched == ref.touched_total(), what
        for x, y in zip(vol, want):
            np.testing.assert_array_equal(x, y, err_msg=what)
        for m in (4, 5):
            for l in range(3):
                np.testing.assert_array_equal(maps(m, l).view(np.uint32), ref.map(m, l).view(np.uint32), err_msg=what)
    for x in (ref, gp, b):
        x.close()


def test_every_count_a_volume_can_hold(kf, oracle32):
    """A snorm16 volume may be uploaded with any count up to 255: the update divides by the count + 1
    and stores at most 128, alike in a single fuse and in a batch's, against the oracle voxel by voxel.
    (Without iterations a batch's session keeps its pose.)"""
    announce("counts 0 to 255")
    seq = small_sequence(seed=12, n_frames=1, w=160, h=120, L=3.0)
    raw = seq.frames(0, 1)[0]
    n, frames = 64, 3
    rng = np.random.default_rng(12)
    Fq = rng.integers(-32768, 32768, n ** 3).astype(np.int16)
    Fq[rng.random(n ** 3) < 0.3] = 32767
    Wq = rng.integers(0, 256, n ** 3).astype(np.uint8)
    grid = kf.VoxelGrid(seq.L, n, mue=0.03, voxel_format=kf.KF_VOXEL_SNORM16_U8)
    b, (sid,) = make_batch(kf, seq, n, 1, iters=(0, 0, 0))
    upload(kf, grid.h, decode_q(Fq), Wq)
    upload(kf, batch_volume(kf, b, sid), decode_q(Fq), Wq)
    dev = kf.DeviceArray.from_host(raw)
    d = oracle32.convert_to_depth_meters(raw, 1e-3)
    dm = kf.GridMap(seq.width, seq.height)
    dm.upload(d)
    sensor = kf.Sensor(seq.fx, seq.fy, seq.cx, seq.cy)
    sensor.set_pose(seq.pose(0))
    above = Wq > 128
    before = Wq.copy()
    for f in range(frames):
        kf.kernel.fuse(dm, grid, sensor)
        b.tick([sid], [dev.ptr.value])
        oracle32.fuse_q(Fq, Wq, n, seq.L, 0.03, d, sensor.get_inverse_pose(), sensor.get_intr(0))
    assert b.status(sid) == 0
    assert np.count_nonzero(above & (Wq != before)) > 1000  # voxels above 128 that the frames met
    for what, (F, W) in [("single", grid.download()), ("batch", b.volume_download(sid))]:
        np.testing.assert_array_equal(W, Wq.astype(np.float32), err_msg=what)
        np.testing.assert_array_equal(F, decode_q(Fq), err_msg=what)
    grid.close()
    b.close()


# ---- the free distances a raycast skips by are formed at the first raycast after a fuse
WALL = dict(n=96, L=2.0, w=160, h=120)


def wall_scene(kf):
    """A camera 0.35 m in front of a 2 m cube and three depth maps of a wall through it: alone, and with
    a box in front of it on the left or on the right (0.9 m away, in what the wall's frames saw as free)."""
    w, h = WALL["w"], WALL["h"]
    sensor = kf.Sensor(0.82 * w, 0.82 * w, w / 2 - 0.5, h / 2 - 0.5)
    pose = np.eye(4, dtype=np.float32)
    pose[3, 2] = -1.35  # column-major
    sensor.set_pose(pose.reshape(-1))
    wall = (1.9 + 0.1 * np.sin(np.arange(w) / 17.0)[None, :] + np.zeros((h, 1))).astype(np.float32)
    left, right = wall.copy(), wall.copy()
    left[h // 4:h // 2, w // 8:w // 3] = 0.9
    right[h // 3:2 * h // 3, 2 * w // 3:5 * w // 6] = 0.9
    return sensor, pose.reshape(-1), [wall, left, right]


def empty_maps(kf):
    init = np.zeros((WALL["h"], WALL["w"], 4), np.float32)
    init[..., 3] = -2
    maps = [kf.GridMap(WALL["w"], WALL["h"], 4) for _ in range(2)]
    for m in maps:
        m.upload(init)
    return maps


def redrawn(kf, handle, fmt, sensor):
    """The maps of a new volume holding the same voxels: its distances come from the voxels."""
    n = WALL["n"]
    fw = np.empty((n ** 3, 2), np.float32)
    kf.check(kf.lib().kf_volume_download(handle, fw.ctypes.data_as(C.c_void_p)))
    grid = kf.VoxelGrid(WALL["L"], n, mue=0.03, voxel_format=fmt)
    kf.check(kf.lib().kf_volume_upload(grid.h, fw.ctypes.data_as(C.c_void_p)))
    maps = empty_maps(kf)
    kf.kernel.raycast(grid, sensor, *maps, 0)
    grid.close()
    return [m.download() for m in maps]


def assert_drawn(got, want, box, what):
    """box: how many of the pixels show the box rather than the wall (0: none)."""
    for g, r in zip(got, want):
        np.testing.assert_array_equal(g.view(np.uint32), r.view(np.uint32), err_msg=what)
    near = np.count_nonzero((want[0][..., 3] == -1) & (want[0][..., 2] < -0.3))
    assert near == 0 if box == 0 else near > box, (what, near)


class Graph:
    """What `record` enqueues on the stream, as a graph."""

    def __init__(self, kf, stream, record):
        self.lib, self.s, self.exec = kf.lib(), stream, C.c_void_p()
        g = C.c_void_p()
        assert self.lib.hipStreamBeginCapture(stream, 0) == 0
        record()
        assert self.lib.hipStreamEndCapture(stream, C.byref(g)) == 0
        assert self.lib.hipGraphInstantiate(C.byref(self.exec), g, None, None, C.c_size_t(0)) == 0
        assert self.lib.hipGraphDestroy(g) == 0

    def replay(self):
        assert self.lib.hipGraphLaunch(self.exec, self.s) == 0
        assert self.lib.hipStreamSynchronize(self.s) == 0

    def close(self):
        assert self.lib.hipGraphExecDestroy(self.exec) == 0


@pytest.mark.parametrize("route", ["eager", "captured fuses", "captured raycasts"])
@pytest.mark.parametrize("fmt", [0, 1])
def test_raycast_after_any_fuse(kf, route, fmt):
    """Boxes that appear where earlier frames saw free space are drawn, whether the fuses, the raycasts or
    neither run from a graph that was captured before.  (Graphs hold launches in pairs: the counters of a
    launch are cleared by the one after it.)"""
    sensor, _, depths = wall_scene(kf)
    lib, n = kf.lib(), WALL["n"]
    grid = kf.VoxelGrid(WALL["L"], n, mue=0.03, voxel_format=fmt)
    stream = C.c_void_p()
    kf.check(lib.kf_stream_create(C.byref(stream)))
    dm = kf.GridMap(WALL["w"], WALL["h"])
    maps = empty_maps(kf)
    sp = C.byref(sensor.s)

    def fuses(times=8):
        for _ in range(times):
            kf.check(lib.kf_fuse(dm.ptr, dm.width, dm.height, grid.h, sp, stream, None))

    def casts():
        for _ in range(2):
            kf.check(lib.kf_raycast(grid.h, sp, maps[0].ptr, maps[1].ptr, dm.width, dm.height, 0, stream, None))

    dm.upload(depths[0])
    fuses(2)
    casts()
    kf.check(lib.kf_stream_synchronize(stream))
    graph = None
    if route != "eager":
        graph = Graph(kf, stream, fuses if route == "captured fuses" else casts)
    for k, times in enumerate([1, 4, 20]):  # left, right, left: each time enough to outweigh what was seen before
        announce(f"raycast after fuses, {route}, format {fmt}, step {k}")
        dm.upload(depths[1 + k % 2])
        for _ in range(times):
            graph.replay() if route == "captured fuses" else fuses()
        kf.check(lib.kf_stream_synchronize(stream))
        graph.replay() if route == "captured raycasts" else casts()
        kf.check(lib.kf_stream_synchronize(stream))
        want = redrawn(kf, grid.h, fmt, sensor)
        assert_drawn([m.download() for m in maps], want, 100, f"{route} step {k}")
    if graph:
        graph.close()
    grid.close()
    kf.check(lib.kf_stream_destroy(stream))


@pytest.mark.parametrize("route", ["batch", "loop", "visualisation volume"])
@pytest.mark.parametrize("fmt", [0, 1])
def test_next_frame_after_a_single_fuse(kf, route, fmt):
    """A program's own kf_fuse into the volume of a batch's session or of the frame loop is seen by the
    next frame's predicted maps, and a volume that is only fused into is drawn as it is when it is
    rendered.  Without iterations the pose stays."""
    sensor, pose, depths = wall_scene(kf)
    lib, n, w, h = kf.lib(), WALL["n"], WALL["w"], WALL["h"]
    raw = kf.DeviceArray.from_host((1000.0 * depths[0]).astype(np.uint16))
    dm = kf.GridMap(w, h)
    icp = kf.IcpConfig((0, 0, 0), w, h, 0.1, TH)
    fx, cx, cy = 0.82 * w, w / 2 - 0.5, h / 2 - 0.5
    handle = C.c_void_p()
    if route == "batch":
        b = kf.Batch(1, icp=icp)
        sid = b.add(kf.SessionConfig(w, h, fx, fx, cx, cy, 1e-3, n, WALL["L"], 0.03, fmt, pose))
        handle = batch_volume(kf, b, sid)
        frame, get, end = lambda: b.tick([sid], [raw.ptr.value]), lambda m: b.map(sid, m), b
    else:
        vis = (n, WALL["L"], 0.03) if route == "visualisation volume" else None
        p = kf.Pipeline(w, h, fx, fx, cx, cy, 1e-3, n, WALL["L"], 0.03, voxel_format=fmt, initial_pose=pose, icp=icp,
                        vis_volume=vis)
        kf.check(lib.kf_pipeline_volume(p.h, C.byref(handle)))
        frame, get, end = lambda: p.frame(raw.ptr.value), p.map, p
    for k in range(3):
        announce(f"single fuse between frames, {route}, format {fmt}, step {k}")
        frame()
        kf.check(lib.kf_device_synchronize())
        if route == "visualisation volume":
            # both volumes saw the same frames: the picture is the tracking volume's
            img = p.render(shading=False)
            maps = empty_maps(kf)
            kf.check(lib.kf_raycast(handle, C.byref(sensor.s), maps[0].ptr, maps[1].ptr, w, h, 0, None, None))
            want = redrawn(kf, handle, fmt, sensor)
            assert_drawn([m.download() for m in maps], want, 0, f"{route} {k}")
            drawn = kf.DeviceArray((h, w), np.uint32)
            inv = np.ascontiguousarray(np.eye(3, dtype=np.float32).reshape(9))
            kf.check(lib.kf_render_normals(maps[1].ptr, w, h, inv.ctypes.data_as(C.c_void_p), drawn.ptr, None, None))
            kf.check(lib.kf_device_synchronize())
            np.testing.assert_array_equal(img, drawn.download())
            assert len(np.unique(img)) > 10
            continue
        dm.upload(depths[1 + k % 2])
        for _ in range((6, 40, 200)[k]):  # enough to outweigh what was seen before
            kf.check(lib.kf_fuse(dm.ptr, w, h, handle, C.byref(sensor.s), None, None))
        kf.check(lib.kf_device_synchronize())
        want = redrawn(kf, handle, fmt, sensor)
        frame()
        kf.check(lib.kf_device_synchronize())
        assert_drawn([get(4), get(5)], want, 100, f"{route} {k}")
    end.close()


# ---- a batch's sweep of bricks in free space
def free_space_bricks(raw_m, n, L, mue, K, cam_z):
    """Bricks (x, y, z) that a camera at (0, 0, cam_z), unturned, certainly updates whole by f = 1: the box
    around the brick's bounding sphere lies in the image with a pixel to spare, the sphere lies between
    the distance limits, and the smallest depth of the 16x16 tiles (64x64 where the box is 48 pixels or
    more) the box touches is more than mue and 2 mm behind it."""
    h, w = raw_m.shape
    d = np.where(np.isfinite(raw_m) & (raw_m > 0), raw_m, 0.0).astype(np.float64)

    def tile_min(s):
        th, tw = -(-h // s), -(-w // s)
        return np.array([[d[y * s:(y + 1) * s, x * s:(x + 1) * s].min() for x in range(tw)] for y in range(th)])

    mins = {16: tile_min(16), 64: tile_min(64)}
    res, r = L / (n - 1), 3.5 * 3 ** 0.5 * L / (n - 1) * 1.01 + 1e-4
    c = -L / 2 + (8 * np.arange(n // 8) + 3.5) * res
    out = np.zeros((n // 8,) * 3, bool)
    for k, z in enumerate(c - cam_z):
        lo, hi = z - r, z + r
        if lo <= 0.402 or hi >= 5.998:
            continue
        for j, y in enumerate(c):
            for i, x in enumerate(c):
                u = [K[0] * f(a / q for q in (lo, hi)) + K[6] + m for f, a, m in ((min, x - r, -2), (max, x + r, 2))]
                v = [K[4] * f(a / q for q in (lo, hi)) + K[7] + m for f, a, m in ((min, y - r, -2), (max, y + r, 2))]
                if u[0] < 0 or v[0] < 0 or u[1] > w - 1 or v[1] > h - 1:
                    continue
                size = max(u[1] - u[0], v[1] - v[0])
                s = 16 if size < 46 else 64
                if size >= 190:
                    continue
                t = mins[s][int(v[0]) // s:int(v[1]) // s + 1, int(u[0]) // s:int(u[1]) // s + 1]
                out[i, j, k] = t.min() - hi >= mue + 2e-3
    return out


@pytest.mark.parametrize("n,w,h", [(200, 320, 240), (96, 200, 148)])
@pytest.mark.parametrize("graph", [False, True])
def test_free_space_sweep_bit_exact(kf, oracle32, n, w, h, graph):
    """A batch updates bricks in free space without projecting their voxels, and only the counts of those
    whose every code is 1: a wall seen over a box that comes and goes, with holes and infinite depths, into
    a volume of uploaded codes and counts (126 to 128 and above among them), so that bricks of every kind
    lie in free space; voxels, fused-voxel counts and the maps drawn from them against the oracle.  (The
    single fuse of the same frames has no such path.)"""
    L, mue, cam_z = 2.0, 0.03, -1.35
    rng = np.random.default_rng(n)
    nb = n // 8
    blow = lambda a: np.repeat(np.repeat(np.repeat(a, 8, 0), 8, 1), 8, 2).reshape(-1)  # noqa: E731
    kind = rng.integers(0, 4, (nb, nb, nb))  # [z, y, x] bricks: untouched, all 1, mixed codes, mixed codes below 0.991
    Fq, Wq = oracle32.new_volume_q(n)
    every = blow(kind)
    for k, codes in [(1, [32767]), (2, [32767, 32767, 32767, 32766, 32471]), (3, [32767, 20000, 3, 0, -500, -32768])]:
        at = every == k
        Fq[at] = rng.choice(np.array(codes, np.int16), int(at.sum()))
        Wq[at] = rng.choice(np.array([0, 1, 5, 126, 127, 128, 129, 200, 255], np.uint8), int(at.sum()))
    sensor = kf.Sensor(0.82 * w, 0.82 * w, w / 2 - 0.5, h / 2 - 0.5)
    pose = np.eye(4, dtype=np.float32)
    pose[3, 2] = cam_z  # column-major
    sensor.set_pose(pose.reshape(-1))
    K, Ki = sensor.get_intr(0), sensor.get_inverse_intr(0)
    b = kf.Batch(1, icp=kf.IcpConfig((0, 0, 0), w, h, 0.1, TH), use_graph=graph)
    sid = b.add(kf.SessionConfig(w, h, 0.82 * w, 0.82 * w, w / 2 - 0.5, h / 2 - 0.5, 1e-3, n, L, mue,
                                 kf.KF_VOXEL_SNORM16_U8, pose.reshape(-1)))
    upload(kf, batch_volume(kf, b, sid), decode_q(Fq), Wq)
    touched, seen = 0, np.zeros(4, int)
    for f in range(5):
        announce(f"free-space sweep n {n} {w}x{h} graph {graph} tick {f}")
        raw = (1900 + 100 * np.sin(np.arange(w) / 17.0)[None, :] + 50 * rng.random((h, w))).astype(np.uint16)
        if f % 2:
            raw[h // 4:h // 2, w // 4:w // 2] = 900
        raw[rng.random((h, w)) < 2e-4] = 0
        raw[3 * h // 4, : w // 3] = 65535
        d = oracle32.convert_to_depth_meters(raw, 1e-3)
        free = free_space_bricks(d, n, L, mue, K, cam_z).transpose(2, 1, 0)
        if f == 0:
            for k in range(4):
                seen[k] = np.count_nonzero(free & (kind == k))
        want = None
        if f:
            init = np.zeros((h, w, 4), np.float32)
            init[..., 3] = -2
            want = oracle32.raycast_q(Fq, n, L, mue, sensor.get_pose(), Ki, w, h, init.copy(), init.copy())
        dev = kf.DeviceArray.from_host(raw)
        b.tick([sid], [dev.ptr.value])
        b.sync()
        touched += oracle32.fuse_q(Fq, Wq, n, L, mue, d, sensor.get_inverse_pose(), K)
        if f:
            for m, x in zip((4, 5), want):
                np.testing.assert_array_equal(b.map(sid, m).view(np.uint32), x.view(np.uint32), err_msg=f"map {m} {f}")
    assert b.status(sid) == 0
    assert (seen > 0).all(), seen  # bricks of every kind met the free-space rule in the first tick
    F, W = b.volume_download(sid)
    np.testing.assert_array_equal(W, Wq.astype(np.float32))
    np.testing.assert_array_equal(F, decode_q(Fq))
    assert b.touched_total() == touched > 0.1 * n ** 3
    b.close()


# ---- volumes of more than 64 bricks a side: two words of free bits per row of bricks
@pytest.mark.parametrize("n", [520, 528])
@pytest.mark.parametrize("fmt", [0, 1])
def test_surface_between_bricks_63_and_64(kf, oracle32, n, fmt):
    """A wall that crosses the plane between bricks 63 and 64 along x, fused where earlier frames saw free
    space, through single fuses and a batch: every voxel and what is drawn against the oracle.  A free bit
    that is not cleared in either word lets a raycast step over the wall."""
    L, mue, w, h = 4.0, 0.03, 160, 120
    # the camera at (-0.5, 0, 0) looks along +x: camera axes x, y, z are -z, y, x of the world
    pose = np.zeros((4, 4), np.float32)
    pose[0, 2], pose[1, 1], pose[2, 0], pose[3] = -1.0, 1.0, 1.0, (-0.5, 0.0, 0.0, 1.0)
    sensor = kf.Sensor(131.25, 131.25, 79.5, 59.5)
    sensor.set_pose(pose.reshape(-1))
    K, Ki = sensor.get_intr(0), sensor.get_inverse_intr(0)
    edge = int(round(1000 * (-L / 2 + 511.5 * L / (n - 1) + 0.5)))  # its depth in millimetres
    u, v = np.meshgrid(np.arange(w), np.arange(h))
    wall = (edge + 60 * np.sin(u / 23.0) * np.cos(v / 19.0)).astype(np.uint16)
    frames = [np.full((h, w), 2900, np.uint16)] + [wall] * 3
    cast, fuse = (oracle32.raycast_q, oracle32.fuse_q) if fmt else (oracle32.raycast, oracle32.fuse)
    Fo, Wo = oracle32.new_volume_q(n) if fmt else oracle32.new_volume(n)
    grid = kf.VoxelGrid(L, n, mue=mue, voxel_format=fmt)
    b = kf.Batch(1, icp=kf.IcpConfig((0, 0, 0), w, h, 0.1, TH))
    sid = b.add(kf.SessionConfig(w, h, 131.25, 131.25, 79.5, 59.5, 1e-3, n, L, mue, fmt, pose.reshape(-1)))
    dm, maps = kf.GridMap(w, h), [kf.GridMap(w, h, 4) for _ in range(2)]
    init = np.zeros((h, w, 4), np.float32)
    init[..., 3] = -2
    for f, raw in enumerate(frames):
        announce(f"wall at bricks 63/64 n {n} format {fmt} frame {f}")
        want = cast(Fo, n, L, mue, sensor.get_pose(), Ki, w, h, init.copy(), init.copy())
        for m in maps:
            m.upload(init)
        kf.kernel.raycast(grid, sensor, *maps, 0)
        dev = kf.DeviceArray.from_host(raw)
        b.tick([sid], [dev.ptr.value])
        b.sync()
        for m, got, x in zip((4, 5), maps, want):
            np.testing.assert_array_equal(got.download().view(np.uint32), x.view(np.uint32), err_msg=f"single {m} {f}")
            if f:
                np.testing.assert_array_equal(b.map(sid, m).view(np.uint32), x.view(np.uint32), err_msg=f"batch {m} {f}")
        d = oracle32.convert_to_depth_meters(raw, 1e-3)
        dm.upload(d)
        kf.kernel.fuse(dm, grid, sensor)
        fuse(Fo, Wo, n, L, mue, d, sensor.get_inverse_pose(), K)
    hit = want[0][..., 3] == -1
    brick = ((want[0][..., 0] + L / 2) / (L / (n - 1)) / 8).astype(int)
    assert np.count_nonzero(hit & (brick == 63)) > 500 and np.count_nonzero(hit & (brick == 64)) > 500
    F, W = (decode_q(Fo), Wo.astype(np.float32)) if fmt else (Fo, Wo)
    for what, (x, y) in [("single", grid.download()), ("batch", b.volume_download(sid))]:
        assert np.array_equal(x.view(np.uint32), F.view(np.uint32)), what
        assert np.array_equal(y.view(np.uint32), W.view(np.uint32)), what
    grid.close()
    b.close()


@pytest.mark.parametrize("degrees", [5.0, 20.0, 60.0, 120.0])
def test_angle_near_the_threshold_bit_exact(kf, oracle32, degrees):
    """The angle test is decided from an approximation except near the threshold: target normals whose
    cosine with the turned live normal lies 2^-25 to 2^-13 to either side of the threshold's, so inside,
    at and outside the band that is evaluated exactly, every row against the oracle's."""
    w, h = 64, 48
    rng = np.random.default_rng(int(degrees))
    f = 60.0
    u, v = np.meshgrid(np.arange(w) + 0.5, np.arange(h) + 0.5)
    z = 1.0 + 0.3 * rng.random((h, w))
    V = np.stack([(u - w / 2) / f * z, (v - h / 2) / f * z, z, np.full((h, w), -1.0)], -1).astype(np.float32)
    live = oracle32.create_normal_map(V)
    th = float(np.float32(np.deg2rad(degrees)))
    accepted = 0
    for turn in range(3):
        announce(f"angle near {degrees} degrees, rotation {turn}")
        Q = np.linalg.qr(rng.standard_normal((3, 3)))[0]
        Q *= np.sign(np.linalg.det(Q))
        R = np.ascontiguousarray(Q.T.reshape(-1), np.float32)  # column-major
        t = rng.standard_normal(3).astype(np.float32)
        a = live[..., :3].astype(np.float64) @ R.reshape(3, 3).astype(np.float64)
        a /= np.maximum(np.linalg.norm(a, axis=-1, keepdims=True), 1e-30)
        side = np.cross(a, rng.standard_normal(a.shape))
        side /= np.maximum(np.linalg.norm(side, axis=-1, keepdims=True), 1e-30)
        c = np.cos(th) + rng.choice([-1.0, 1.0], (h, w)) * 2.0 ** rng.uniform(-25, -13, (h, w))
        N = c[..., None] * a + np.sqrt(1 - c * c)[..., None] * side
        TN = np.concatenate([N, np.full((h, w, 1), -1.0)], -1).astype(np.float32)
        TV = np.concatenate([rng.standard_normal((h, w, 3)), np.full((h, w, 1), -1.0)], -1).astype(np.float32)
        maps = []
        for m in (V, TV, TN):
            g = kf.GridMap(w, h, 4)
            g.upload(m)
            maps.append(g)
        K = np.array([f, 0, 0, 0, f, 0, w / 2, h / 2, 1], np.float32)
        A, b = kf.DeviceArray((h * w, 6)), kf.DeviceArray((h * w,))
        kf.kernel.construct_icp_residuals(*maps, R, t, R, t, K, 1e18, th, A, b)
        Ar, br = oracle32.construct_icp_residuals(V, TV, TN, R, t, R, t, K, 1e18, th)
        np.testing.assert_array_equal(A.download().view(np.uint32), Ar.view(np.uint32))
        np.testing.assert_array_equal(b.download().view(np.uint32), br.view(np.uint32))
        hits = np.count_nonzero(np.any(Ar != 0, axis=1))
        accepted += hits
        _, inliers = kf.kernel.icp_reduce(*maps, R, t, R, t, K, 1e18, th)
        assert inliers == hits
    assert 0.2 < accepted / (3 * (w - 1) * (h - 1)) < 0.8


# voxels much longer than a step of the march: a box of free bricks holds many times the march's range
@pytest.mark.parametrize("n,L,mue", [(8, 9000.0, 1e-3), (16, 2000.0, 0.03), (64, 400.0, 0.01), (128, 1024.0, 0.5)])
def test_raycast_of_long_voxels_bit_exact(kf, oracle32, n, L, mue):
    """Random voxels, drawn from places where the rays' few metres cross the plane where F changes sign, lie
    in free space or behind the surface, against the oracle."""
    w, h = 64, 48
    rng = np.random.default_rng(n)
    res = L / n
    F = (0.992 + 0.008 * rng.random((n, n, n), np.float32)).astype(np.float32)
    F[n // 2:] = -(0.2 + 0.8 * rng.random((n - n // 2, n, n), np.float32))  # z
    F[n // 2 - 1] = 0.2 + 0.8 * rng.random((n, n), np.float32)
    grid = kf.VoxelGrid(L, n, mue=mue)
    grid.upload(F.reshape(-1), np.ones(n ** 3, np.float32))
    sensor = kf.Sensor(60.0, 60.0, w / 2 - 0.5, h / 2 - 0.5)
    maps = [kf.GridMap(w, h, 4) for _ in range(2)]
    init = np.zeros((h, w, 4), np.float32)
    init[..., 3] = -2
    hits = 0
    # F at the middle column between the voxel planes either side of the change of sign
    col = F[n // 2 - 1:n // 2 + 1, n // 2 - 1:n // 2 + 1, n // 2 - 1:n // 2 + 1].mean((1, 2)).astype(np.float64)
    zero = -0.5 * res + res * col[0] / (col[0] - col[1])
    for k, z in enumerate([zero - 2.5, zero - 5.0, zero + 1.0, -0.3 * L, -0.5 * L - 1.0]):
        pose = np.eye(4, dtype=np.float32)
        pose[3, 2] = z  # column-major
        sensor.set_pose(pose.reshape(-1))
        announce(f"raycast of long voxels n {n} L {L} mue {mue} pose {k}")
        for m in maps:
            m.upload(init)
        kf.kernel.raycast(grid, sensor, *maps, 0)
        want = oracle32.raycast(F.reshape(-1), n, L, mue, sensor.get_pose(), sensor.get_inverse_intr(0), w, h,
                                init.copy(), init.copy())
        hits += np.count_nonzero(want[0][..., 3] == -1)
        for m, x in zip(maps, want):
            np.testing.assert_array_equal(m.download().view(np.uint32), x.view(np.uint32), err_msg=f"pose {k}")
    assert hits > 500
    grid.close()


@pytest.mark.parametrize("dist", [-1.0, -0.0, 0.0, 1e-25, 1e-3, 0.05, 1e18, 1e20, float("inf"), float("nan")])
def test_any_distance_threshold_bit_exact(kf, oracle32, dist):
    """The distance test takes any threshold: none is met by a length above it, a negative one by no
    length at all, 0 by coincident points, an infinite one by every length; targets at, near and 1e20 m
    from the vertices, some of them infinite or NaN, every row against the oracle's."""
    w, h = 64, 48
    rng = np.random.default_rng(7)
    f = 60.0
    u, v = np.meshgrid(np.arange(w) + 0.5, np.arange(h) + 0.5)
    z = 1.0 + 0.1 * rng.random((h, w))
    V = np.stack([(u - w / 2) / f * z, (v - h / 2) / f * z, z, np.full((h, w), -1.0)], -1).astype(np.float32)
    TV = V.copy()
    kind = rng.integers(0, 6, (h, w))
    for k, size in [(1, 1e-4), (2, 0.05), (3, 3.0), (4, 1e20)]:
        at = kind == k
        TV[at, :3] += (size * rng.standard_normal((int(at.sum()), 3))).astype(np.float32)
    odd = (kind == 5) & (rng.random((h, w)) < 0.2)
    TV[odd, 0] = rng.choice(np.array([np.inf, -np.inf, np.nan], np.float32), int(odd.sum()))
    N = np.concatenate([0.1 * rng.standard_normal((h, w, 2)), np.ones((h, w, 1))], -1)
    TN = np.concatenate([N / np.linalg.norm(N, axis=-1, keepdims=True), np.full((h, w, 1), -1.0)], -1)
    TN = TN.astype(np.float32)
    maps = []
    for m in (V, TV, TN):
        g = kf.GridMap(w, h, 4)
        g.upload(m)
        maps.append(g)
    R, t = np.eye(3, dtype=np.float32).reshape(9), np.zeros(3, np.float32)
    K = np.array([f, 0, 0, 0, f, 0, w / 2, h / 2, 1], np.float32)
    A, b = kf.DeviceArray((h * w, 6)), kf.DeviceArray((h * w,))
    for degrees in (60.0, 180.0):
        announce(f"distance threshold {dist}, {degrees} degrees")
        th = float(np.float32(np.deg2rad(degrees)))
        kf.kernel.construct_icp_residuals(*maps, R, t, R, t, K, dist, th, A, b)
        Ar, br = oracle32.construct_icp_residuals(V, TV, TN, R, t, R, t, K, dist, th)
        for got, want in ((A.download(), Ar), (b.download(), br)):
            nan = np.isnan(want)
            np.testing.assert_array_equal(np.isnan(got), nan)
            np.testing.assert_array_equal(np.where(nan, 0, got.view(np.uint32)), np.where(nan, 0, want.view(np.uint32)))
        kept = np.count_nonzero(np.any(Ar != 0, axis=1) | (br != 0))  # NaN differs from 0
        _, inliers = kf.kernel.icp_reduce(*maps, R, t, R, t, K, dist, th)
        assert inliers == kept


def test_maps_of_a_loop_that_still_runs(kf, oracle32):
    """Pipeline.map returns the last enqueued frame's map without a sync before it, also the normals, which
    are formed when they are asked for: with frames in flight, the normals of the vertices, level by level."""
    seq = small_sequence(seed=14, n_frames=4, w=640, h=480, L=4.0)
    raws = seq.frames(0, 4)
    dev = kf.DeviceArray.from_host(raws)
    p = make_pipeline(kf, seq, 256, 0)
    for rep in range(3):
        announce(f"maps of a running loop {rep}")
        for f in range(4):
            p.frame(dev.ptr.value + f * raws[0].nbytes)
        for l in range(3):
            n, v = p.map(3, l), p.map(2, l)
            d = p.map(1, l)
            np.testing.assert_array_equal(n.view(np.uint32), oracle32.create_normal_map(v).view(np.uint32))
            if l == 0:
                want = oracle32.apply_bilateral_filter(oracle32.convert_to_depth_meters(raws[3], 1e-3))
                np.testing.assert_array_equal(d.view(np.uint32), want.view(np.uint32))
    p.close()
