"""ops.graph_capture: no cyclic garbage is collected while a graph is captured."""
import contextlib
import gc

import torch

from loqa_hub_amd import ops


def test_collector_is_off_during_captures(monkeypatch):
    seen = []

    @contextlib.contextmanager
    def graph(g, **kw):
        seen.append((g, kw))
        yield
    monkeypatch.setattr(torch.cuda, "graph", graph)
    assert gc.isenabled()
    with ops.graph_capture("a", pool=1):
        assert not gc.isenabled()
        with ops.graph_capture("b"):
            assert not gc.isenabled()
        assert not gc.isenabled()
    assert gc.isenabled() and seen == [("a", {"pool": 1}), ("b", {})]
    try:
        with ops.graph_capture("c"):
            raise ValueError
    except ValueError:
        pass
    assert gc.isenabled()
    gc.disable()
    try:
        with ops.graph_capture("d"):
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()
