"""Grids and trees whose kernels need more threads than one launch may have
(2^32 along an axis): a plane of 2^32 voxels, and a level of 2^24 nodes."""
import numpy as np
import pytest

from oracle import xo
from xenodon_amd import abi

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(300)]

SIDE = 1 << 16


@pytest.fixture(scope="module")
def plane():
    """65536 x 65536 x 1 voxels, a few of them coloured, the last among them; 2^28 bricks."""
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    grid = np.zeros((1, SIDE, SIDE, 4), np.uint8)
    at = [(SIDE - 1, SIDE - 1), (SIDE - 1, SIDE - 2), (SIDE - 3, 5), (SIDE // 2, SIDE - 1)]  # y, x
    for k, (y, x) in enumerate(at):
        grid[0, y, x] = (200, 40 + 50 * k, 90, 255)
    with abi.Context(0) as ctx:
        yield ctx, grid, ctx.grid_volume(grid), at


def test_bricks_of_a_plane_of_2_32_voxels(plane):
    ctx, grid, vol, at = plane
    ov = xo.OracleVolume(grid=grid)
    for y, x in at:
        eye = ((x + 0.5) / SIDE, (y + 0.5) / SIDE, -4.0 / SIDE)
        cam = (0.0, 0.0, 1.0), (0.0, 1.0, 0.0), eye
        args = (31, 31, [SIDE, SIDE, 1])
        got, _ = ctx.render_image(vol, abi.DDA, abi.make_camera(*cam), abi.make_uniforms(*args, emission=3e4))
        want = xo.render(abi.DDA, ov, xo.make_camera(*cam), xo.make_uniforms(*args, emission=3e4))["rgba"]
        assert want[..., :3].any()
        assert np.array_equal(got, want), (y, x)


def test_a_level_too_large_to_scan_is_refused(plane):
    """Every node of a plane is split down to the voxels: 2^31 nodes of 2 voxels a side, more than the scans count."""
    ctx, _, vol, _ = plane
    for tree in (abi.TREE_SPARSE, abi.TREE_DAG):
        with pytest.raises(abi.XdError) as err:
            ctx.build_octree(vol, tree=tree)
        assert err.value.status == abi.XD_ERR_FORMAT


def test_statistics_of_2_28_bricks():
    """4096 x 2048 x 2048 voxels, a few of them coloured: the tree down to each of these from the root, and every other
    leaf empty."""
    grid = np.zeros((2048, 2048, 4096, 4), np.uint8)
    at = [(4095, 2047, 2047), (0, 0, 2047), (4094, 3, 1029), (2047, 2047, 0)]  # x, y, z
    for k, (x, y, z) in enumerate(at):
        grid[z, y, x] = (200, 40 + 50 * k, 90, 255)
    with abi.Context(0) as ctx:
        nodes, st = ctx.build_octree(ctx.grid_volume(grid))
    assert st["side"] == 4096
    leaf = nodes[:, 9] >= 1 << 31
    seen = {0}
    for x, y, z in at:
        i = 0
        for d in range(12):
            assert not leaf[i] and nodes[i, 9] == d
            i = int(nodes[i, (x >> (11 - d) & 1) << 2 | (y >> (11 - d) & 1) << 1 | (z >> (11 - d) & 1)])
            seen.add(i)
        assert nodes[i, 9] == 0x8000000C and nodes[i, 8] == grid[z, y, x].view(np.uint32)[0]
    assert len(nodes) == 1 + 8 * sum(not leaf[i] for i in seen)
    leaf[list(seen)] = False
    assert not nodes[leaf, 8].any()


def test_standard_deviation_of_a_level_of_2_24_nodes():
    """32768 x 16384 x 8 voxels: nodes of 16 voxels a side reach out of the grid and are split, 8 into each.  Of those
    some hold two colours, far enough apart for either heuristic, so the two give one tree."""
    grid = np.zeros((8, 16384, 32768, 4), np.uint8)
    rng = np.random.default_rng(3)
    for x, y in [(4095, 2047), (0, 0)] + [(rng.integers(4096), rng.integers(2048)) for _ in range(60)]:
        grid[:, 8 * y:8 * y + 8, 8 * x:8 * x + 4] = rng.integers(100, 256, 4)
    with abi.Context(0) as ctx:
        vol = ctx.grid_volume(grid)
        want, _ = ctx.build_octree(vol, heuristic=abi.HEURISTIC_CHAN_DIFF, chan_diff=20)
        got, _ = ctx.build_octree(vol, heuristic=abi.HEURISTIC_STD_DEV, std_dev=5.0)
    level = got[:, 9] & 0xFF
    assert (level == 12).sum() >= 1 << 24 and (level == 13).any()
    assert np.array_equal(got, want)
