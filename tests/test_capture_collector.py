"""Captures and the cyclic collector: nothing that died before is freed while one is open (a graph's own end may not run there)."""
import contextlib
import gc
import threading

import pytest
import torch

from umbrella_amd import _lib


class Graph:
    def register_generator_state(self, generator):
        self.registered_in_mode = torch.is_inference_mode_enabled()


class Dead:
    """stands in a cycle, as an engine and its target do; says on its end whether a capture was open"""
    def __init__(self, log, open_):
        self.me, self.log, self.open = self, log, open_

    def __del__(self):
        self.log.append(self.open[0])


@pytest.fixture
def stand_in(monkeypatch):
    open_ = [0]

    @contextlib.contextmanager
    def graph(g, **kw):
        open_[0] += 1
        try:
            yield
        finally:
            open_[0] -= 1
    monkeypatch.setattr(torch.cuda, "graph", graph)
    monkeypatch.setattr(torch.cuda, "default_generators", (None,))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    was = gc.isenabled()
    yield open_
    (gc.enable if was else gc.disable)()


def _allocate():
    kept = [[i] for i in range(3 * gc.get_threshold()[0] * gc.get_threshold()[1])]      # past the first two generations' thresholds
    return len(kept)


@pytest.mark.parametrize("on", [True, False])
@pytest.mark.parametrize("fails", [True, False])
def test_nothing_is_freed_inside(stand_in, on, fails):
    (gc.enable if on else gc.disable)()
    log = []
    Dead(log, stand_in)
    with pytest.raises(KeyError) if fails else contextlib.nullcontext():
        with _lib.capturing(Graph()):
            _allocate()
            assert not gc.isenabled()
            if fails:
                raise KeyError("body")
    assert not any(log) and gc.isenabled() == on
    gc.collect()
    assert log == [0]


def test_captures_of_two_threads(stand_in):
    """the second ends behind the first: the collector comes back with the last one only"""
    gc.enable()
    entered, leave, seen = threading.Event(), threading.Event(), []

    def other():
        with _lib.capturing(Graph()):
            entered.set()
            leave.wait(20)
            seen.append(gc.isenabled())
    t = threading.Thread(target=other)
    with _lib.capturing(Graph()):
        t.start()
        assert entered.wait(20)
    assert not gc.isenabled()
    leave.set()
    t.join()
    assert seen == [False] and gc.isenabled()


@pytest.mark.parametrize("inference", [True, False])
@pytest.mark.parametrize("grad", [True, False])
def test_the_body_runs_in_the_modes_of_the_caller(stand_in, inference, grad):
    g = Graph()
    with torch.inference_mode(inference), torch.set_grad_enabled(grad):
        with _lib.capturing(g):
            assert torch.is_inference_mode_enabled() == inference and torch.is_grad_enabled() == grad
        assert torch.is_inference_mode_enabled() == inference and torch.is_grad_enabled() == grad
    assert g.registered_in_mode is False
