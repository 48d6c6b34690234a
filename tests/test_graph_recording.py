"""Recording a decode step, with stand-ins for the device's graphs: nothing is destroyed by the cyclic collector meanwhile."""
import contextlib
import gc
import threading
import types

import pytest
import torch

from llm_sharding_amd.runtime.engine import DecodeGraph


class DeadGraph:
    """A captured graph in a cycle: its end is noted with what was going on then."""

    def __init__(self, log, state):
        self.me, self.log, self.state = self, log, state

    def __del__(self):
        self.log.append(self.state["recording"])


@pytest.fixture
def device(monkeypatch):
    """torch.cuda's streams and graphs without a device; ["recording"]: inside a capture."""
    state = {"recording": False}

    @contextlib.contextmanager
    def graph(g, stream=None):
        state["recording"] = True
        try:
            yield
        finally:
            state["recording"] = False
    stream = types.SimpleNamespace(wait_stream=lambda s: None)
    monkeypatch.setattr(torch.cuda, "Stream", lambda device=None: stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: object())
    monkeypatch.setattr(torch.cuda, "graph", graph)
    was, at = gc.isenabled(), gc.get_threshold()
    gc.set_threshold(50, 2, 2)
    gc.enable()
    yield state
    gc.set_threshold(*at)
    (gc.enable if was else gc.disable)()


def _step(body):
    g = object.__new__(DecodeGraph)
    g.eng = types.SimpleNamespace(device=torch.device("cpu"), carries_state=False)
    g.pos, g.tokens, g.keys, g.step_ctr = (torch.zeros(2, dtype=torch.int32) for _ in range(4))
    g.history = g.pre_comm = g.post_comm = None
    g.split_head = False
    g._body = body
    return g


def test_nothing_is_collected_while_a_step_is_recorded(device):
    log = []

    def body():  # what a step does on the host: many short-lived objects, after a graph was dropped in a cycle
        DeadGraph(log, device)
        for _ in range(20):
            [[] for _ in range(200)]
    _step(body).capture(warmup=False)
    assert True not in log
    [[] for _ in range(2000)]  # ... and the collector runs again
    gc.collect()
    assert log == [False] and gc.isenabled()


def test_a_step_that_raises_gives_the_collector_back(device):
    def body():
        assert not gc.isenabled()
        raise RuntimeError("step")
    with pytest.raises(RuntimeError, match="step"):
        _step(body).capture(warmup=False)
    assert gc.isenabled()


def test_overlapping_recordings_and_a_collector_that_was_off(device):
    from llm_sharding_amd.runtime.recording import collector_held
    inside, leave = threading.Event(), threading.Event()

    def other():
        with collector_held():
            inside.set()
            leave.wait(30)
    t = threading.Thread(target=other)
    t.start()
    assert inside.wait(30)
    with collector_held():
        pass
    assert not gc.isenabled()  # the other one still records
    leave.set()
    t.join(30)
    assert gc.isenabled()
    gc.disable()
    with collector_held():
        pass
    assert not gc.isenabled()
