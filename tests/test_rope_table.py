"""The rotary table is shared by all ops of a process: it is complete before another stream or thread can find it."""
import types

import pytest
import torch

from eet_amd import ops


def test_complete_before_it_is_shared(monkeypatch):
    events = []

    def build(*args):
        events.append("launch")
        return 0

    def synchronize():
        assert not ops._rope_tables, "in the cache while its kernel may still run"
        events.append("wait")
    monkeypatch.setattr(ops, "_rope_tables", {})
    monkeypatch.setattr(ops, "lib", lambda: types.SimpleNamespace(eet_rope_table=build))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: types.SimpleNamespace(synchronize=synchronize))
    table = ops._rope_table(3, 4, "cpu")
    assert events == ["launch", "wait"] and ops._rope_table(3, 4, "cpu") is table


@pytest.mark.gpu
def test_read_from_another_stream(gpu, monkeypatch):
    """Built behind other work, read at once from a stream that does not wait for that."""
    want = ops._rope_table(777, 64, gpu).clone()
    monkeypatch.setattr(ops, "_rope_tables", {})
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    a = torch.randn(4096, 4096, device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        for _ in range(20):
            a @ a
        table = ops._rope_table(777, 64, gpu)
    with torch.cuda.stream(other):
        got = table.clone()
    other.synchronize()
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_recorded_into_a_graph(gpu, monkeypatch):
    """A table that a graph builds is not handed to anyone else: before a replay it holds nothing."""
    want = ops._rope_table(55, 96, gpu).clone()
    monkeypatch.setattr(ops, "_rope_tables", {})
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        table = ops._rope_table(55, 96, gpu)
    assert not ops._rope_tables
    for _ in range(3):
        table.zero_()
        graph.replay()
        assert torch.equal(table, want)
