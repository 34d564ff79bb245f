"""Frame readback through the pinned ring: frames below, at and above a slot
(1 MiB) and the ring (16 MiB), whole and into wider host rows, rows longer than
a slot among them, hold the pixels that small renders of the same regions give."""
import ctypes

import numpy as np
import pytest

from tests import helpers as H
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

# width, height: one pixel; under a slot; a slot exactly; ragged over a slot; over the ring; rows over a slot
SIZES = [(1, 1), (199, 143), (512, 512), (1021, 1031), (2500, 1999), (300001, 3)]


@pytest.mark.parametrize("W,Hh", SIZES)
@pytest.mark.parametrize("pad", [0, 5])
def test_download_sizes_and_strides(W, Hh, pad):
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    with abi.Context(0) as ctx:
        vol = ctx.grid_volume(H.random_grid((8, 8, 8), density=1.0, seed=4))
        cam = abi.make_camera(*H.look_at((0.5, 0.4, 0.5), (0.9, 0.6, 0.3)))
        fr = ctx.frame(W, Hh)
        ctx.render(vol, abi.DDA, cam, abi.make_uniforms(W, Hh, [8] * 3, emission=1.5), fr)
        got = np.full((Hh, W + pad), 0x01020304, np.uint32)
        abi.check(abi.lib().xd_frame_download(fr.h, ctypes.c_void_p(got.ctypes.data), W + pad))
        assert (got[:, W:] == 0x01020304).all()
        img = np.ascontiguousarray(got[:, :W]).view(np.uint8).reshape(Hh, W, 4)
        assert np.array_equal(img, fr.download())
        # regions of the same display, small enough for one slot
        for x0, y0 in {(0, 0), (max(0, W - 64), max(0, Hh - 48)), (W // 2, Hh // 2)}:
            w, h = min(64, W - x0), min(48, Hh - y0)
            part, _ = ctx.render_image(vol, abi.DDA, cam, abi.make_uniforms(
                w, h, [8] * 3, emission=1.5, out_offset=(x0, y0), disp_extent=(W, Hh)))
            assert np.array_equal(img[y0:y0 + h, x0:x0 + w], part)


def test_download_waits_for_the_null_stream():
    """A program that works on a frame's device memory on the null stream gets what that work wrote."""
    hip = abi.lib()  # finds the HIP runtime's functions as well
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipMemsetAsync.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t, ctypes.c_void_p]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    size = 4 << 30
    with abi.Context(0) as ctx:
        fr = ctx.frame(640, 360)
        buf = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(buf), size) == 0
        for value in (3, 200):
            for _ in range(8):  # some milliseconds
                assert hip.hipMemsetAsync(buf, value, size, None) == 0
            assert hip.hipMemsetAsync(fr.device_ptr(), value, 640 * 360 * 4, None) == 0
            assert (fr.download() == value).all()
        hip.hipFree(buf)
