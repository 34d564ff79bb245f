"""A frame's device memory is the program's too: what it has queued there on the null
stream ends before the renders that follow a set of views or the load of an octree."""
import ctypes

import numpy as np
import pytest

from tests import helpers as H
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

W, HH = 64, 48
BUSY = 4 << 30


@pytest.fixture(scope="module")
def env():
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    hip = abi.lib()  # finds the HIP runtime's functions as well
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipMemsetAsync.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t, ctypes.c_void_p]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    with abi.Context(0) as ctx:
        buf = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(buf), BUSY) == 0

        def write_late(frame):
            for value in range(8):  # some milliseconds
                assert hip.hipMemsetAsync(buf, value, BUSY, None) == 0
            assert hip.hipMemsetAsync(frame.device_ptr(), 7, W * HH * 4, None) == 0

        yield ctx, write_late
        hip.hipFree(buf)


CAM = abi.make_camera(*H.look_at((0.5, 0.4, 0.5), (0.9, 0.6, 0.3)))


def test_batch_views(env):
    ctx, write_late = env
    vol = ctx.grid_volume(H.random_grid((24, 24, 24), density=1.0, seed=3))
    view = (vol, abi.DDA, CAM, abi.make_uniforms(W, HH, [24] * 3, emission=1.5))
    want, _ = ctx.render_image(*view)
    frame, b = ctx.frame(W, HH), ctx.batch()
    for _ in range(3):
        write_late(frame)
        b.set_views([view + (frame,)])
        b.render()
        assert np.array_equal(frame.download(), want)
    b.free()


@pytest.mark.parametrize("tree", [abi.TREE_SPARSE, abi.TREE_DAG])  # derived on the device; on the host
@pytest.mark.parametrize("layout", [0, 1, 2])
def test_octree_load(env, tree, layout):
    ctx, write_late = env
    nodes, st = abi.build_octree(H.random_grid((24, 24, 24), density=1.0, seed=3), tree=tree)
    uni = abi.make_uniforms(W, HH, [st["side"]] * 3, emission=1.5)
    vol = ctx.svo_volume(nodes, st["side"])
    want, _ = ctx.render_image(vol, abi.ESVO, CAM, uni)
    vol.free()
    frame = ctx.frame(W, HH)
    ctx.set_option("octree_layout", layout)
    try:
        write_late(frame)
        vol = ctx.svo_volume(nodes, st["side"])
    finally:
        ctx.set_option("octree_layout", 0)
    ctx.render(vol, abi.ESVO, CAM, uni, frame)
    assert np.array_equal(frame.download(), want)
    vol.free()
