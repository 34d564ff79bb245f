"""Octree upload: the layout derived on the device (and, for what it does not
take, on the host) gives the frames of the .svo words as they are, for trees at
the edges of its blocks and for node orders and shapes that no converter writes."""
import numpy as np
import pytest

from tests import helpers as H
from xenodon_amd import abi

pytestmark = pytest.mark.gpu

LEAF = 0x80000000
OCTREE = [abi.SVO_NAIVE, abi.ESVO, abi.SVO_DF, abi.SVO_ROPE]


@pytest.fixture(scope="module")
def ctx():
    if abi.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    c = abi.Context(0)
    yield c
    c.close()


def random_tree(parents, seed, max_depth=6):
    """.svo nodes of a random tree of `parents` internal nodes in pre-order (children after their parent)."""
    rng = np.random.default_rng(seed)
    # the shape first: which nodes are internal, breadth-first growth
    kids, depth, leaves = {}, {0: 0}, [0]
    n = 1
    for _ in range(parents):
        open_ = [i for i in leaves if depth[i] < max_depth]
        p = open_[rng.integers(len(open_))]
        leaves.remove(p)
        kids[p] = list(range(n, n + 8))
        for c in kids[p]:
            depth[c] = depth[p] + 1
            leaves.append(c)
        n += 8
    order, stack = [], [0]
    while stack:
        i = stack.pop()
        order.append(i)
        stack += kids.get(i, [])
    at = {old: new for new, old in enumerate(order)}
    nodes = np.zeros((n, 10), np.uint32)
    for old, new in at.items():
        colour = 0 if rng.random() < 0.3 else int(rng.integers(1, 1 << 24)) | 0xFF000000
        nodes[new, 8], nodes[new, 9] = colour, depth[old] | (0 if old in kids else LEAF)
        if old in kids:
            nodes[new, :8] = [at[c] for c in kids[old]]
    return nodes


def _frames(ctx, nodes, layout, travs=OCTREE, side=64):
    ctx.set_option("octree_layout", layout)
    try:
        vol = ctx.svo_volume(nodes, side)
    finally:
        ctx.set_option("octree_layout", 0)
    out = []
    for f, up, eye in H.orbit_cameras(2, 1.5, seed=9) + [H.look_at((0.4, 0.6, 0.45), (0.9, 0.1, 0.8))]:
        for t in travs:
            uni = abi.make_uniforms(53, 41, [side] * 3, emission=1.2)
            out.append(ctx.render_image(vol, t, abi.make_camera(f, up, eye), uni)[0])
    info = vol.info()
    vol.free()
    return out, (info.max_depth, info.is_rope, info.node_count)


def _same(ctx, nodes, travs=OCTREE):
    ref, ref_info = _frames(ctx, nodes, 1, travs)
    for layout in (0, 2):
        got, info = _frames(ctx, nodes, layout, travs)
        assert info == ref_info
        for a, b in zip(got, ref):
            assert np.array_equal(a, b), layout
    return ref


# 512 nodes a block: 505, 513 and 521 nodes straddle the first edge
@pytest.mark.parametrize("parents", [0, 1, 2, 9, 63, 64, 65, 640])
def test_trees_at_block_edges(ctx, parents):
    _same(ctx, random_tree(parents, seed=parents))


def test_leaf_root_with_a_depth_field(ctx):
    nodes = np.zeros((1, 10), np.uint32)
    nodes[0, 8], nodes[0, 9] = 0xFF30A060, LEAF | 3
    _same(ctx, nodes)


@pytest.mark.parametrize("kind", ["rope", "sparse", "dag"])
def test_converter_trees(ctx, kind):
    grid = H.random_grid((23, 37, 30), density=0.2, seed=4)
    nodes, _ = abi.build_octree(grid, tree={"rope": abi.TREE_ROPE, "sparse": abi.TREE_SPARSE, "dag": abi.TREE_DAG}[kind])
    assert any(img[..., :3].any() for img in _same(ctx, nodes))


def test_shuffled_order_orphans_shared_children_and_inexact_depths(ctx):
    rng = np.random.default_rng(8)
    base = random_tree(70, seed=8)
    n = len(base)
    # nodes in any order, the root first
    at = np.concatenate([[0], 1 + rng.permutation(n - 1)]).astype(np.uint32)
    shuffled = np.zeros_like(base)
    shuffled[at] = base
    inner = (shuffled[:, 9] & LEAF) == 0
    shuffled[inner, :8] = at[shuffled[inner, :8]]
    _same(ctx, shuffled)
    # nodes that nothing names: eight leaves, and an internal node with them as children
    leaf = np.zeros((8, 10), np.uint32)
    leaf[:, 9] = LEAF | 3
    _same(ctx, np.concatenate([base, leaf]))
    extra = np.zeros((1, 10), np.uint32)
    extra[0, :8], extra[0, 9] = n + 1 + np.arange(8), 2
    _same(ctx, np.concatenate([base, extra, leaf]))
    # a child named twice, and so a node named by none, at a node count that a tree could have
    shared = base.copy()
    p = int(np.flatnonzero((base[:, 9] & LEAF) == 0)[-1])
    shared[p, 3] = shared[p, 5]
    _same(ctx, shared)
    # a depth field that is not the node's depth (svo-df and svo-rope read it)
    inexact = base.copy()
    inexact[p, 9] += 1
    _same(ctx, inexact)


def test_malformed_nodes_are_refused(ctx):
    for bad in ("child", "cycle", "depth"):
        nodes = random_tree(20, seed=3)
        inner = np.flatnonzero((nodes[:, 9] & LEAF) == 0)
        p = int(inner[-1])
        if bad == "child":
            nodes[p, 2] = len(nodes)
        elif bad == "cycle":
            nodes[p, 2] = 0
        else:
            nodes[p, 9] = 65
        with pytest.raises(abi.XdError) as err:
            ctx.svo_volume(nodes, 64)
        assert err.value.status == abi.XD_ERR_FORMAT


@pytest.mark.parametrize("level", [0, 1, 2])
def test_internal_children_named_twice_near_the_root(ctx, level):
    """All children of a node of the first levels are one internal child, the others and what is below them named by
    none: a node count that a tree could have, but more child words to number than there are nodes."""
    nodes = random_tree(600, seed=1)
    inner = (nodes[:, 9] & LEAF) == 0
    p = 0
    for _ in range(level):
        p = next(int(c) for c in nodes[p, :8] if inner[c])
    nodes[p, :8] = next(int(c) for c in nodes[p, :8] if inner[c])
    _same(ctx, nodes)
