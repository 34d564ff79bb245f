"""The device octree builder against the host converter, node for node, where
its pieces meet: boxes that end inside a brick, a statistics cell or a block of
cells, single voxels, std-dev sums of one part and of many, and limits that the
sums reach exactly."""
import numpy as np
import pytest

from tests import helpers as H
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

# x, y, z
DIMS = [(1, 1, 1), (3, 1, 2), (4, 4, 4), (5, 9, 17), (33, 16, 8), (64, 64, 64), (130, 21, 7), (65, 70, 129)]


@pytest.fixture(scope="module")
def ctx():
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    c = abi.Context(0)
    yield c
    c.close()


def _grid(dims):
    """Noise over smooth ramps, with a flat region and an empty one."""
    x, y, z = dims
    rng = np.random.default_rng(sum(dims))
    Z, Y, X = np.meshgrid(np.arange(z), np.arange(y), np.arange(x), indexing="ij")
    g = np.stack([X * 3, Y * 5, (X + Z) * 2, 40 + 0 * X], -1) % 256
    g = (g + rng.integers(0, 6, g.shape)) % 256
    g[: z // 2, : y // 2, : x // 2] = 77
    g[z // 2:, y // 2:, x // 2:] = 0
    return g.astype(np.uint8)


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("kind", [abi.TREE_SPARSE, abi.TREE_ROPE, abi.TREE_DAG])
def test_builder_edges(ctx, dims, kind):
    grid = _grid(dims)
    gv = ctx.grid_volume(grid)
    settings = [(abi.HEURISTIC_CHAN_DIFF, c, 0.0) for c in (0, 9, 255)] + \
               [(abi.HEURISTIC_STD_DEV, 0, s) for s in (0.0, 2.5, 12.0, 1e9)]
    for heuristic, chan, sd in settings:
        want, wst = abi.build_octree(grid, heuristic=heuristic, chan_diff=chan, std_dev=sd, tree=kind)
        got, gst = ctx.build_octree(gv, heuristic=heuristic, chan_diff=chan, std_dev=sd, tree=kind)
        assert gst == wst, (heuristic, chan, sd)
        assert np.array_equal(got, want), (heuristic, chan, sd)
    gv.free()


def test_std_dev_limit_reached_exactly(ctx):
    """Half the voxels at 0 and half at 2d: sqrt(S / n) is d * sqrt(channels), and a limit of just that does not split."""
    grid = np.zeros((32, 32, 32, 4), np.uint8)
    grid[::2] = 20
    gv = ctx.grid_volume(grid)
    for sd in (np.nextafter(20.0, 0), 20.0, np.nextafter(20.0, 99)):
        want, wst = abi.build_octree(grid, heuristic=abi.HEURISTIC_STD_DEV, std_dev=float(sd))
        got, gst = ctx.build_octree(gv, heuristic=abi.HEURISTIC_STD_DEV, std_dev=float(sd))
        assert gst == wst and np.array_equal(got, want), sd
    gv.free()


# x, y, z: a node of the upper levels is mostly outside of these
THIN = [(2, 4099, 4), (1, (1 << 17) + 1, 6), (70000, 3, 2), (5, 1, 1 << 18), (1, 1030, 517)]


@pytest.mark.parametrize("dims", THIN)
def test_std_dev_of_thin_grids(ctx, dims):
    """The sums take the grid's part of a node, not the side^3 of all of it."""
    x, y, z = dims
    grid = np.random.default_rng(x + y).integers(0, 256, (z, y, x, 4), dtype=np.uint8)
    gv = ctx.grid_volume(grid)
    for sd in (100.0, 140.0, 150.0):
        want, wst = abi.build_octree(grid, heuristic=abi.HEURISTIC_STD_DEV, std_dev=sd)
        got, gst = ctx.build_octree(gv, heuristic=abi.HEURISTIC_STD_DEV, std_dev=sd)
        assert gst == wst, sd
        assert np.array_equal(got, want), sd
    gv.free()


def test_side_limit(ctx):
    """Node codes hold 21 levels: a grid of 2^21 voxels a side is converted, a longer one refused."""
    line = np.zeros((1, 1, (1 << 21) + 1, 4), np.uint8)
    gv = ctx.grid_volume(line[:, :, :-1])
    nodes, st = ctx.build_octree(gv)
    assert st["side"] == 1 << 21 and len(nodes) == 1 + 8 * ((1 << 21) - 1)
    gv.free()
    gv = ctx.grid_volume(line)
    with pytest.raises(abi.XdError) as err:
        ctx.build_octree(gv)
    assert err.value.status == abi.XD_ERR_FORMAT
    gv.free()
