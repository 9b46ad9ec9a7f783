"""kf_session_bytes (host arithmetic): what a session is charged in HBM covers its places in the
batch's shared lists."""
import ctypes as C

import pytest


def charged(w, h, n, fmt):
    from kfusion import SessionConfig, _capi
    b = C.c_size_t()
    assert _capi.load().kf_session_bytes(C.byref(SessionConfig(w, h, volume_n=n, voxel_format=fmt)), C.byref(b)) == 0
    return b.value


def held(w, h):
    """Of a w x h frame: metres, filtered depth, three maps of 16 bytes a pixel on three levels, the
    depth ranges of 16x16 and 64x64 tiles, and two sets of 64-float partial rows for the most
    workgroups of 256 lanes a level takes (one pixel a lane at these sizes)."""
    up = lambda a, b: -(-a // b)  # noqa: E731
    px = [(w >> l) * (h >> l) for l in range(3)]
    return (8 * px[0] + 48 * sum(px) + 8 * (up(w, 16) * up(h, 16) + up(w, 64) * up(h, 64)) +
            2 * 4 * 64 * max(up(p, 256) for p in px))


def ray_places(w, h):
    """A level's 8x8 tiles come in multiples of 8, one band per XCD; a place is a ray of 32 bytes."""
    return sum(64 * 8 * -(-(-(-(w >> l) // 8) * -(-(h >> l) // 8)) // 8) for l in range(3))


@pytest.mark.parametrize("w,h", [(100, 76), (64, 48), (4, 4), (76, 52), (160, 120)])
@pytest.mark.parametrize("fmt", [0, 1])
def test_a_session_is_charged_its_places_in_the_ray_lists(w, h, fmt):
    """Against a frame of whole tiles (256x256: 1024, 256 and 64): the charges differ by what the
    sessions hold and by their rays' places in the lists of both formats, which grow 2x at a time."""
    assert ray_places(256, 256) == 64 * (1024 + 256 + 64)
    rays = 2 * 2 * 32 * (ray_places(256, 256) - ray_places(w, h))
    assert charged(256, 256, 64, fmt) - charged(w, h, 64, fmt) == held(256, 256) - held(w, h) + rays
