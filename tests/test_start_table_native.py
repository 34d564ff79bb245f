"""The start table in the order, the coarseness and with the flags that the kernels
read (csrc/xd_table.hpp), entry for entry against the plain table, on the host
(tests/native/table_check.cpp): every shift from single leaves to nine levels."""
import os
import subprocess

import numpy as np
import pytest

from oracle import xo
from tests import helpers as H
from xenodon_amd import build as native_build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("table") / "table_check")
    cmd = [native_build.hipcc(), "-O2", "-std=c++17", "-pthread", "-I", native_build.INCLUDE, "-I", native_build.CSRC,
           os.path.join(HERE, "native", "table_check.cpp"), os.path.join(native_build.CSRC, "xd_layout.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return out


@pytest.mark.parametrize("levels, wide", [(k, "0") for k in range(10)] + [(2, "1"), (9, "1")])
def test_device_table_equals_the_plain_one(harness, tmp_path, levels, wide):
    side = 1 << levels
    grid = np.zeros((min(side, 24), min(side, 20), side, 4), np.uint8)  # z, y, x
    part = H.random_grid((grid.shape[0], grid.shape[1], min(side, 40)), density=0.4, seed=levels)
    grid[:, :, :part.shape[2]] = part
    nodes, _ = xo.build_octree(grid, tree=xo.TREE_DAG if levels == 6 else xo.TREE_SPARSE)
    path = tmp_path / "tree.words"
    np.ascontiguousarray(nodes, dtype=np.uint32).tofile(path)
    r = subprocess.run([harness, str(path), wide], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-1000:]
    assert f"depth {levels}" in r.stdout
    assert ("low cells 1" in r.stdout) == (levels > 8)
