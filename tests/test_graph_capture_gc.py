"""No cycle is collected inside a capture of decode graphs: what a dropped engine
held is gone before, and the collector is off until the captures are done."""
import contextlib
import gc
import types
import weakref

import pytest
import torch

from gpustack_amd.engine.graph_runner import DecodeGraphRunner


class _Cycle:
    def __init__(self):
        self.me = self


@pytest.mark.parametrize("fails", [False, True])
def test_the_collector_is_off_while_graphs_are_captured(monkeypatch, fails):
    for name, f in (("graph_pool_handle", lambda: None),
                    ("synchronize", lambda *a: None), ("CUDAGraph", object),
                    ("graph", lambda *a, **k: contextlib.nullcontext())):
        monkeypatch.setattr(torch.cuda, name, f)
    gc.disable()                  # the cycle lives until capture asks for it
    old = weakref.ref(_Cycle())
    assert old() is not None
    gc.enable()
    seen = []

    def model(*a, **k):
        seen.append((gc.isenabled(), old() is None))
        if fails:
            raise RuntimeError("refused")

    runner = DecodeGraphRunner.__new__(DecodeGraphRunner)
    runner.runner = types.SimpleNamespace(model=model, kv=None)
    runner.buckets, runner.want_hidden = [1, 2], False
    runner.tokens = torch.zeros(2, dtype=torch.long)
    runner.graphs, runner.outs, runner.metas = {}, {}, {}
    runner._meta = lambda bs: None
    with pytest.raises(RuntimeError) if fails else contextlib.nullcontext():
        runner.capture()
    assert seen and all(s == (False, True) for s in seen)
    assert gc.isenabled()
