"""The batched forms' tile queues: launches from one wave tile up to more tiles
than resident waves, growing and shrinking on one batch object (whose captured
launch is reused), give the plain render's frames, bit for bit."""
import ctypes

import numpy as np
import pytest

from tests import helpers as H
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

TRAVERSALS = [abi.DDA, abi.SVO_NAIVE, abi.ESVO, abi.SVO_DF, abi.SVO_ROPE]
# (views, width, height): 1 tile; one block; a few blocks; ~13000 tiles; small again
SHAPES = [(1, 1, 1), (4, 8, 8), (5, 37, 29), (40, 161, 127), (2, 9, 8), (15, 64, 65)]


@pytest.fixture(scope="module")
def env():
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    ctx = abi.Context(0)
    grid = H.blocky_grid(32, 4, seed=5)
    nodes, st = abi.build_octree(grid, tree=abi.TREE_ROPE)
    yield ctx, (ctx.grid_volume(grid), [32] * 3), (ctx.svo_volume(nodes, st["side"]), [st["side"]] * 3)
    ctx.close()


@pytest.mark.parametrize("travs", [[t] for t in TRAVERSALS] + [TRAVERSALS])
@pytest.mark.parametrize("class_kernels,waves,grab", [(0, 8, 1), (1, 0, 4)])
def test_queue_sizes_match_plain_renders(env, travs, class_kernels, waves, grab):
    ctx, grid, svo = env
    b = ctx.batch()
    b.set_tuning([8] * 5, tiles_per_grab=grab, waves_per_simd=waves, class_kernels=class_kernels)
    for n, W, Hh in SHAPES:
        views = []
        for k, (f, up, eye) in enumerate(H.orbit_cameras(n, 1.6, seed=n)):
            t = travs[k % len(travs)]
            vol, md = grid if t == abi.DDA else svo
            views.append((vol, t, abi.make_camera(f, up, eye), abi.make_uniforms(W, Hh, md, emission=1.5),
                          ctx.frame(W, Hh)))
        refs = [ctx.render_image(*v[:4])[0] for v in views]
        b.set_views(views)
        for _ in range(2):
            b.render()
            for v, ref in zip(views, refs):
                assert np.array_equal(v[4].download(), ref), (n, W, Hh)
        abi.render_static(ctx, views, {"tile_w": [8] * 5, "class_kernels": class_kernels})
        for v, ref in zip(views, refs):
            assert np.array_equal(v[4].download(), ref), (n, W, Hh, "static")
            v[4].free()
    b.free()


@pytest.mark.parametrize("order", [0, 2, 3, 4])
@pytest.mark.parametrize("tile_w,rpl", [(8, 1), (16, 2), (32, 4)])
def test_every_tile_is_dealt(env, order, tile_w, rpl):
    """Every pixel of views cut into whole, narrow and low squares is rendered: the frames are black before, and
    every ray inside this volume is lit."""
    ctx, _, _ = env
    grid = H.random_grid((24, 24, 24), density=1.0, seed=3)
    vol = ctx.grid_volume(grid)
    away = abi.make_camera(*H.look_at((0.5, 0.5, 3.0), (0.5, 0.5, 9.0)))
    views = []
    for k, (W, Hh) in enumerate([(8, 8), (65, 8), (8, 65), (129, 57), (520, 24), (24, 520), (333, 222), (1, 700)]):
        fr = ctx.frame(W, Hh)
        uni = abi.make_uniforms(W, Hh, [24] * 3, emission=2.0)
        ctx.render(vol, abi.DDA, away, uni, fr)
        assert not fr.download()[..., :3].any()
        views.append((vol, abi.DDA, abi.make_camera(*H.look_at((0.5, 0.45, 0.55), (0.2 + 0.1 * k, 0.5, 0.1))), uni, fr))
    b = ctx.batch()
    b.set_tuning([tile_w] * 5, interleave=order, rays_per_lane=[rpl] * 5)
    b.set_views(views)
    b.render()
    for v in views:
        got = v[4].download()
        assert got[..., :3].any(-1).all()
        assert np.array_equal(got, ctx.render_image(*v[:4])[0])
        v[4].free()
    b.free()
    vol.free()


@pytest.mark.parametrize("travs", [[abi.DDA], [abi.SVO_DF], TRAVERSALS])
@pytest.mark.parametrize("class_kernels", [0, 1])
def test_queue_sizes_on_frames_that_hold_something_else(env, travs, class_kernels):
    """Each launch alone fills its frames: before it they hold bytes that no frame has (a pixel's last is 255)."""
    ctx, grid, svo = env
    hip = abi.lib()  # finds the HIP runtime's functions as well
    hip.hipMemset.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t]
    b = ctx.batch()
    b.set_tuning([8] * 5, class_kernels=class_kernels)
    for n, W, Hh in SHAPES:
        views = []
        for k, (f, up, eye) in enumerate(H.orbit_cameras(n, 1.6, seed=n)):
            t = travs[k % len(travs)]
            vol, md = grid if t == abi.DDA else svo
            views.append((vol, t, abi.make_camera(f, up, eye), abi.make_uniforms(W, Hh, md, emission=1.5),
                          ctx.frame(W, Hh)))
        refs = [ctx.render_image(*v[:4])[0] for v in views]
        b.set_views(views)
        for launch in (b.render, b.render,
                       lambda: abi.render_static(ctx, views, {"tile_w": [8] * 5, "class_kernels": class_kernels})):
            for v in views:
                assert hip.hipMemset(v[4].device_ptr(), 0x55, W * Hh * 4) == 0
                assert (v[4].download() == 0x55).all()
            launch()
            for v, ref in zip(views, refs):
                assert np.array_equal(v[4].download(), ref), (n, W, Hh)
        for v in views:
            v[4].free()
    b.free()
