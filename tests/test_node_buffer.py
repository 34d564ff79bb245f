"""The converter's node array is the library's own buffer: it lives as long as a
view of it, into the interpreter's exit handlers."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = """
import atexit
held = []
atexit.register(lambda: print("sum", int(held[0].sum(dtype='uint64'))))
import numpy as np
from xenodon_amd import abi
grid = np.random.default_rng(3).integers(0, 256, (32, 32, 32, 4), dtype=np.uint8)
nodes, stats = abi.build_octree(grid, tree=abi.TREE_SPARSE)
held.append(nodes[5:])
print("sum", int(held[0].sum(dtype='uint64')))
"""


def test_nodes_live_into_exit_handlers():
    r = subprocess.run([sys.executable, "-c", CODE], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    first, last = r.stdout.split("\n")[:2]
    assert first.startswith("sum ") and first == last
