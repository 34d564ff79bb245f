"""A context that goes together with its volumes, frames, batches and servers (in a
reference cycle, or with a program's globals at exit) releases them once, whatever
order the collector takes them in."""
import gc

import pytest

from xenodon_amd import abi


class Recorder:
    """Stands in for the native library: which handles were released after their context."""

    def __init__(self):
        self.closed, self.late = set(), []

    def __getattr__(self, name):
        def call(h=None, *args):
            if name == "xd_close":
                self.closed.add(h)
            elif name.endswith("_free") and h[0] in self.closed:
                self.late.append((name, h))
            return abi.XD_OK
        return call


@pytest.mark.parametrize("first", [False, True])
def test_children_in_a_cycle_with_their_context(monkeypatch, first):
    rec = Recorder()
    monkeypatch.setattr(abi, "lib", lambda: rec)

    def build():
        made = []
        if first:  # the collector meets the children before their context, too
            made += [object.__new__(cls) for cls in (abi.Volume, abi.Frame, abi.Batch, abi.Server)]
        ctx = abi.Context(0)
        ctx.h = "ctx"
        if not first:
            made += [object.__new__(cls) for cls in (abi.Volume, abi.Frame, abi.Batch, abi.Server)]
        for k, c in enumerate(made):
            c.ctx, c.h = ctx, ("ctx", k)
            ctx._adopt(c)
        cycle = {"ctx": ctx, "children": made}
        cycle["self"] = cycle

    build()
    gc.collect()
    assert rec.closed == {"ctx"}
    assert rec.late == []
