"""Mapping through every route that fuses or draws a volume (single calls, the frame loop, batch ticks):
frames that are not fused, uploaded states, volumes of more than 64 bricks a side."""
import numpy as np
import pytest

from gpu_util import announce, small_sequence

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
