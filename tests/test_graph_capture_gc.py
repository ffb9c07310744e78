"""Captured graphs that only the cyclic collector can free (a runner whose function refers back to it) must not be
freed while another graph is being captured: destroying a graph synchronises the device, which a capture forbids,
and an error raised there ends the process. CPU, with stand-ins for the stream and graph objects."""
import contextlib
import gc
import threading

import pytest
import torch

from torchair_amd import graph as tai_graph


class _Stream:
    def __init__(self, device=None):
        pass

    def wait_stream(self, other):
        pass


@pytest.fixture
def fake_cuda(monkeypatch):
    """Stand-ins that note the graphs destroyed inside a capture. entering: called as a capture begins."""
    state = {"capturing": 0, "destroyed_inside": 0, "destroyed": 0, "entering": lambda: None}

    class Graph:
        def __del__(self):
            state["destroyed"] += 1
            state["destroyed_inside"] += state["capturing"] > 0

    @contextlib.contextmanager
    def capture(graph):
        state["capturing"] += 1
        state["entering"]()
        try:
            yield
        finally:
            state["capturing"] -= 1

    monkeypatch.setattr(torch.cuda, "Stream", _Stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: _Stream())
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "graph", capture)
    was = gc.get_threshold(), gc.isenabled()
    gc.collect()
    gc.enable()
    yield state
    gc.set_threshold(*was[0])
    gc.enable() if was[1] else gc.disable()


def _capture(fn):
    x = torch.zeros(1)
    return tai_graph._Captured(fn, [x], [True], [True])


def _drop_in_cycle(captured):
    """Leaves the captured graph to the collector: state -> runner -> function -> state."""
    state = {}
    runner = tai_graph.HipGraphRunner(lambda x: (state, x))
    runner.graphs["key"] = captured.pop()
    state["runner"] = runner


def _busy(x):
    """Allocates containers, as the Python of a captured step does; the collector runs on such allocations."""
    keep = [[i] for i in range(3000)]
    return keep and x


def test_the_collector_stays_off_inside_a_capture(fake_cuda):
    first = [_capture(_busy)]

    def entering():  # a runner is dropped, and the collector due at the next few allocations
        _drop_in_cycle(first)
        gc.set_threshold(1, 1, 1)

    before = fake_cuda["destroyed"]
    fake_cuda["entering"] = entering
    kept = _capture(_busy)
    assert not first and fake_cuda["destroyed_inside"] == 0
    assert gc.isenabled()
    gc.set_threshold(700, 10, 10)
    gc.collect()
    assert fake_cuda["destroyed"] == before + 1  # freed outside the capture
    del kept


def test_the_collector_is_restored(fake_cuda):
    """After a failing capture, and left off where the program keeps it off."""
    def fails(x):
        if fake_cuda["capturing"]:
            assert not gc.isenabled()
            raise ValueError("in the capture")
        return x
    with pytest.raises(ValueError, match="in the capture"):
        _capture(fails)
    assert gc.isenabled()
    gc.disable()
    _capture(_busy)
    assert not gc.isenabled()


def test_captures_of_two_threads_overlap(fake_cuda):
    """The collector comes back when the last of two overlapping captures ends, not the first."""
    inside, go_on, seen = threading.Event(), threading.Event(), []

    def slow(x):
        if fake_cuda["capturing"]:
            inside.set()
            go_on.wait(10)
            seen.append(gc.isenabled())
        return x

    def other(x):
        return x

    t = threading.Thread(target=lambda: _capture(slow))
    t.start()
    assert inside.wait(10)
    _capture(other)  # begins and ends inside the other's capture
    seen.append(gc.isenabled())
    go_on.set()
    t.join(10)
    assert seen == [False, False]
    assert gc.isenabled()
