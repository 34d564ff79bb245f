"""The DDA's batches of steps against the oracle, bit for bit, where they can go
wrong: grids of one voxel up to several macro cells with ragged edges, lone
voxels at a batch's reach from the ray, rays that start inside, on a face or far
outside, and a model box larger or smaller than the grid."""
import numpy as np
import pytest

from oracle import xo
from tests import helpers as H
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (4, 9, 3), (8, 8, 8), (17, 16, 15), (40, 24, 33), (260, 6, 5), (7, 5, 140)]  # x, y, z


@pytest.fixture(scope="module")
def ctx():
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    c = abi.Context(0)
    yield c
    c.close()


def _lone_voxels(dims, seed):
    """A few coloured voxels, the corners among them, in an empty grid."""
    rng = np.random.default_rng(seed)
    x, y, z = dims
    g = np.zeros((z, y, x, 4), np.uint8)
    for at in [(0, 0, 0), (z - 1, y - 1, x - 1)] + [tuple(rng.integers(0, (z, y, x))) for _ in range(6)]:
        g[at] = rng.integers(1, 256, 4)
    return g


CAMERAS = H.orbit_cameras(3, 1.7, seed=3) + [
    H.look_at((0.45, 0.55, 0.4), (0.9, 0.2, 0.7)),     # inside
    H.look_at((0.5, 0.5, 0.0), (0.5, 0.5, 1.0)),       # on a face, along an axis
    H.look_at((0.5, 0.5, -1.0), (0.5, 0.5, 1.0)),
    H.look_at((300.0, 200.0, -250.0), (0.5, 0.5, 0.5)),  # far: the entry rounds off the faces
]


@pytest.mark.parametrize("scale", [1.0, 1.7, 0.6])
@pytest.mark.parametrize("dims", DIMS)
def test_dda_runs_match_the_oracle(ctx, dims, scale):
    md = [max(1, int(round(d * scale))) for d in dims]  # the uniform's model box
    for grid in (_lone_voxels(dims, 1), H.random_grid(dims[::-1], density=0.3, seed=2)):
        ov, gv = xo.OracleVolume(grid=grid), ctx.grid_volume(grid)
        views, refs = [], []
        for f, up, eye in CAMERAS:
            ref = xo.render(abi.DDA, ov, xo.make_camera(f, up, eye), xo.make_uniforms(61, 43, md, emission=0.8))["rgba"]
            cam, uni = abi.make_camera(f, up, eye), abi.make_uniforms(61, 43, md, emission=0.8)
            img, _ = ctx.render_image(gv, abi.DDA, cam, uni)
            assert np.array_equal(img, ref), (dims, scale, eye)
            views.append((gv, abi.DDA, cam, uni, ctx.frame(61, 43)))
            refs.append(ref)
        b = ctx.batch()
        for class_kernels in (1, 0):
            b.set_tuning([8] * 5, class_kernels=class_kernels)
            b.set_views(views)
            b.render()
            for v, ref in zip(views, refs):
                assert np.array_equal(v[4].download(), ref), (dims, scale, class_kernels)
        b.free()
        for v in views:
            v[4].free()
        gv.free()


@pytest.mark.parametrize("scale", [1.0, 1.7])
@pytest.mark.parametrize("dims", DIMS)
def test_dda_runs_in_the_kernel_of_all_traversals(ctx, dims, scale):
    """An octree view beside them takes the DDA views to that kernel, whose batches of steps are shorter.  The frames
    hold black before each launch."""
    md = [max(1, int(round(d * scale))) for d in dims]
    grid = _lone_voxels(dims, 1)
    ov, gv = xo.OracleVolume(grid=grid), ctx.grid_volume(grid)
    nodes, st = abi.build_octree(H.blocky_grid(16, 4, seed=5))
    sv = ctx.svo_volume(nodes, st["side"])
    away = abi.make_camera(*H.look_at((0.5, 0.5, 3.0), (0.5, 0.5, 9.0)))
    views, refs = [], []
    for f, up, eye in CAMERAS:
        refs.append(xo.render(abi.DDA, ov, xo.make_camera(f, up, eye), xo.make_uniforms(61, 43, md, emission=0.8))["rgba"])
        views.append((gv, abi.DDA, abi.make_camera(f, up, eye), abi.make_uniforms(61, 43, md, emission=0.8),
                      ctx.frame(61, 43)))
    tree = (sv, abi.ESVO, away, abi.make_uniforms(9, 9, [st["side"]] * 3), ctx.frame(9, 9))
    b = ctx.batch()
    b.set_tuning([8] * 5, class_kernels=0)
    for launch in (lambda: (b.set_views(views + [tree]), b.render()),
                   lambda: abi.render_static(ctx, views + [tree], {"tile_w": [8] * 5, "class_kernels": 0})):
        for v in views:
            ctx.render(gv, abi.DDA, away, v[3], v[4])
            assert not v[4].download()[..., :3].any()
        launch()
        for v, ref in zip(views, refs):
            assert np.array_equal(v[4].download(), ref), (dims, scale)
    b.free()
    for v in views + [tree]:
        v[4].free()
    gv.free()
    sv.free()
