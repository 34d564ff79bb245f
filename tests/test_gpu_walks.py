"""The octree walks that take a short cut (esvo and svo-rope from cell to cell,
svo-df by the four children that a ray passes) against the general walk on the raw node words:
trees at the edges of the short cuts' ranges (1 level; the start table's 8 levels
and one around them; the most levels and one more) and cameras that they must
pass on or that meet cell borders exactly."""
import numpy as np
import pytest

from oracle import xo
from tests.test_gpu_parity import _chain_tree
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

TARGET = (0.3712345, 0.6123457, 0.5317891)
RAW = 1  # octree_layout: the node words as they are, which the general walk reads


@pytest.fixture(scope="module")
def ctx():
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    with abi.Context(0) as c:
        yield c


def _camera(eye, fwd, up=(0.0, 1.0, 0.0)):
    f = np.array(fwd, float) / np.linalg.norm(fwd)
    r = np.cross(up, f)
    r /= np.linalg.norm(r)
    return abi.make_camera(f, np.cross(f, r), eye)


CAMERAS = {
    "towards": lambda: _camera((-0.4, 1.1, -0.7), np.array(TARGET) - (-0.4, 1.1, -0.7)),
    "back": lambda: _camera((1.3, 0.2, 1.6), np.array(TARGET) - (1.3, 0.2, 1.6)),
    "inside": lambda: _camera(np.array(TARGET) + (2e-3, -1e-3, 3e-3), (-2.0, 1.0, -3.0)),
    "axis": lambda: _camera((0.5, 0.5, -1.0), (0.0, 0.0, 1.0)),
    "axis_inside": lambda: _camera((0.375, 0.625, 0.5), (-1.0, 0.0, 0.0)),
    "diagonal": lambda: _camera((-0.5, 0.5, -0.5), (1.0, 0.0, 1.0)),
    "corner": lambda: _camera((0.0, 0.0, 0.0), (1.0, 1.0, 1.0)),
    "face": lambda: _camera((1.0, 0.25, 0.75), (0.0, 1.0, 1e-6)),
    "away": lambda: _camera((-0.4, 1.1, -0.7), (-1.0, 0.2, -1.0)),
    "far": lambda: _camera((3e4, 2e4, -1e4), np.array((0.5, 0.5, 0.5)) - (3e4, 2e4, -1e4)),
}


def _pair(ctx, nodes, side, t, cam, W=97, H=61):
    uni = abi.make_uniforms(W, H, [side] * 3, emission=1.5)
    images = []
    for layout in (0, RAW):
        ctx.set_option("octree_layout", layout)
        try:
            vol = ctx.svo_volume(nodes, side)
        finally:
            ctx.set_option("octree_layout", 0)
        images.append(ctx.render_image(vol, t, cam, uni)[0])
        vol.free()
    return images


def _tree(depth, t, seed):
    nodes = _chain_tree(depth, TARGET, seed=seed)
    if t == abi.SVO_ROPE:
        xo.lib().xo_generate_ropes(nodes.ctypes.data, nodes.shape[0], 1 << depth)
    return nodes


@pytest.mark.parametrize("depth", [1, 2, 7, 8, 9, 10, 12, 13, 14, 15])
@pytest.mark.parametrize("t", [abi.ESVO, abi.SVO_DF, abi.SVO_ROPE])
def test_chain_trees(ctx, t, depth):
    nodes = _tree(depth, t, seed=depth)
    lit = 0
    for name, cam in CAMERAS.items():
        got, want = _pair(ctx, nodes, 1 << depth, t, cam())
        assert np.array_equal(got, want), (name, int((got != want).any(-1).sum()))
        lit += int(want[..., :3].any())
    assert lit >= 6


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 1e30])
@pytest.mark.parametrize("axis", [0, 2])
@pytest.mark.parametrize("t", [abi.ESVO, abi.SVO_DF, abi.SVO_ROPE])
def test_cameras_out_of_range(ctx, t, axis, bad):
    nodes = _tree(9, t, seed=3)
    eye = [0.4, 0.6, -0.8]
    eye[axis] = bad
    got, want = _pair(ctx, nodes, 512, t, _camera(eye, (0.1, 0.05, 1.0)), 33, 17)
    assert np.array_equal(got, want)


def _grid():
    rng = np.random.default_rng(8)
    grid = rng.integers(0, 256, (24, 24, 24, 4), dtype=np.uint8)
    grid[rng.random((24, 24, 24)) < 0.6] = 0
    return np.kron(grid, np.ones((2, 2, 2, 1), np.uint8))


@pytest.mark.parametrize("t, tree", [(abi.ESVO, abi.TREE_DAG), (abi.ESVO, abi.TREE_SPARSE), (abi.SVO_DF, abi.TREE_DAG),
                                     (abi.SVO_DF, abi.TREE_SPARSE), (abi.SVO_ROPE, abi.TREE_ROPE),
                                     (abi.SVO_ROPE, abi.TREE_SPARSE)])
def test_built_trees(ctx, t, tree):
    """Every kind of leaf; the DAG has no records, the sparse tree no ropes."""
    nodes, st = abi.build_octree(_grid(), tree=tree)
    for name, cam in CAMERAS.items():
        got, want = _pair(ctx, nodes, st["side"], t, cam())
        assert np.array_equal(got, want), name


@pytest.mark.parametrize("depth", [8, 10])
@pytest.mark.parametrize("change", ["cut", "turned", "deeper", "higher", "depth"])
def test_changed_ropes(ctx, change, depth):
    """Ropes that do not lead where the geometry says are followed as they are."""
    if depth == 8:  # the grid in a corner of 256^3 voxels
        grid = np.zeros((48, 48, 129, 4), np.uint8)
        grid[:, :, 1:49] = _grid()
        grid[:, :, 128] = 77
        nodes, st = abi.build_octree(grid, tree=abi.TREE_ROPE)
        nodes, side = nodes.copy(), st["side"]
        assert side == 256
    else:
        nodes, side = _tree(depth, abi.SVO_ROPE, seed=5), 1 << depth
    leaf = nodes[:, 9] >= 1 << 31
    parent = np.zeros(len(nodes), np.int64)
    for k in range(8):
        parent[nodes[~leaf, k]] = np.nonzero(~leaf)[0]
    where = np.nonzero(leaf[:, None] & (nodes[:, :6] != 0))
    pick = np.random.default_rng(2).choice(len(where[0]), max(1, len(where[0]) // 7), replace=False)
    for i, k in zip(where[0][pick], where[1][pick]):
        to = nodes[i, k]
        if change == "cut":
            nodes[i, k] = 0
        elif change == "turned":
            nodes[i, k] = nodes[i, (k + 2) % 6]
        elif change == "deeper" and not leaf[to]:
            nodes[i, k] = nodes[to, 3]
        elif change == "higher" and parent[to]:
            nodes[i, k] = parent[to]
        elif change == "depth":
            nodes[i, 9] = (nodes[i, 9] & 0x80000000) | max(1, int(nodes[i, 9] & 0xFF) - 1)
    for name, cam in CAMERAS.items():
        got, want = _pair(ctx, nodes, side, abi.SVO_ROPE, cam(), 41, 29)
        assert np.array_equal(got, want), name


def _corner_tree(depth):
    """A rope tree of blocky voxels in a corner of 2^depth voxels a side, with leaves above the start table's level
    beside regions that reach down to it."""
    block = _grid() if depth == 8 else np.kron(_grid(), np.ones((2, 2, 2, 1), np.uint8))
    size, half = block.shape[0], 1 << (depth - 1)
    grid = np.zeros((size, size, half + 1, 4), np.uint8)
    grid[:, :, :size] = block
    grid[:, :, half] = 77
    nodes, st = abi.build_octree(grid, tree=abi.TREE_ROPE)
    assert st["side"] == 1 << depth
    return nodes.copy(), st["side"], size / st["side"]


@pytest.mark.parametrize("depth", [8, 10])
@pytest.mark.parametrize("to", ["child", "between", "corner"])
def test_ropes_into_the_near_corner_of_their_target(ctx, to, depth):
    """A rope that leads to a descendant at its target's lower corner, which the place beside the leaf is in as well,
    ends in that descendant wherever the ray goes on."""
    nodes, side, used = _corner_tree(depth)
    plain = nodes.copy()
    leaf = nodes[:, 9] >= 1 << 31
    turned = 0
    for i, k in zip(*np.nonzero(leaf[:, None] & (nodes[:, :6] != 0))):
        chain = [nodes[i, k]]
        while not leaf[chain[-1]]:
            chain.append(nodes[chain[-1], 0])
        if nodes[chain[-1], 9] & 0xFF > 8:  # below the table: the place's entry is none of the chain's leaves
            continue
        if to == "between":
            pick = 1 + len(chain[1:-1]) // 2 if len(chain) > 3 else 0
        else:
            pick = min(1, len(chain) - 1) if to == "child" else len(chain) - 1
        nodes[i, k] = chain[pick]
        turned += pick > 0
    assert turned > 20
    mid = 0.5 * used
    near = [_camera((-0.8 * used, 1.4 * used, -1.1 * used), np.array([mid] * 3) - np.array((-0.8, 1.4, -1.1)) * used),
            _camera((2.1 * used, -0.7 * used, 1.3 * used), np.array([mid] * 3) - np.array((2.1, -0.7, 1.3)) * used),
            _camera((0.4 * used, 0.45 * used, 0.7 * used), (1.0, -0.7, -0.4))]
    changed = 0
    for cam in near + [make() for make in CAMERAS.values()]:
        got, want = _pair(ctx, nodes, side, abi.SVO_ROPE, cam, 41, 29)
        changed += int((want != _pair(ctx, plain, side, abi.SVO_ROPE, cam, 41, 29)[1]).any())
        assert np.array_equal(got, want), int((got != want).any(-1).sum())
    assert changed  # or the ropes would not matter to these views


@pytest.mark.parametrize("depth", [1, 2, 7, 8, 9, 10, 12, 14, 22])
def test_naive_chain_trees(ctx, depth):
    nodes = _tree(depth, abi.SVO_NAIVE, seed=depth)
    for name, cam in CAMERAS.items():
        got, want = _pair(ctx, nodes, 1 << depth, abi.SVO_NAIVE, cam())
        assert np.array_equal(got, want), name


@pytest.mark.parametrize("tree", [abi.TREE_SPARSE, abi.TREE_ROPE, abi.TREE_DAG])
def test_naive_built_trees(ctx, tree):
    nodes, st = abi.build_octree(_grid(), tree=tree)
    for name, cam in CAMERAS.items():
        got, want = _pair(ctx, nodes, st["side"], abi.SVO_NAIVE, cam())
        assert np.array_equal(got, want), name


@pytest.mark.parametrize("t, tree", [(t, abi.TREE_ROPE) for t in (abi.SVO_NAIVE, abi.ESVO, abi.SVO_DF, abi.SVO_ROPE)] +
                         [(t, abi.TREE_DAG) for t in (abi.SVO_NAIVE, abi.ESVO, abi.SVO_DF)])
def test_wide_tags_below_the_start_table(ctx, t, tree):
    """31-bit indices without an empty tag, in trees of 10 levels: leaves and records below the table's 8."""
    nodes, side, used = _corner_tree(10)
    if tree == abi.TREE_DAG:
        block = np.kron(_grid(), np.ones((2, 2, 2, 1), np.uint8))
        grid = np.zeros((96, 96, 513, 4), np.uint8)
        grid[:, :, 1:97] = block
        nodes, st = abi.build_octree(grid, tree=tree)
        side = st["side"]
    vols = []
    for layout in (RAW, 2):
        ctx.set_option("octree_layout", layout)
        try:
            vols.append(ctx.svo_volume(nodes, side))
        finally:
            ctx.set_option("octree_layout", 0)
    mid = 0.5 * used
    near = [_camera((-0.8 * used, 1.4 * used, -1.1 * used), np.array([mid] * 3) - np.array((-0.8, 1.4, -1.1)) * used),
            _camera((0.4 * used, 0.45 * used, 0.7 * used), (1.0, -0.7, -0.4))]
    for cam in near + [make() for make in CAMERAS.values()]:
        uni = abi.make_uniforms(61, 47, [side] * 3, emission=1.5)
        want, got = (ctx.render_image(v, t, cam, uni)[0] for v in vols)
        assert np.array_equal(got, want)
    for v in vols:
        v.free()
