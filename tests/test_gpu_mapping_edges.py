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
