"""Recording a decode step and dropping what holds recorded ones, with stand-ins for the device's graphs: nothing is destroyed by the
cyclic collector while a step is recorded, and product objects that hold graphs die when the last reference to them goes."""
import contextlib
import gc
import threading
import types
import weakref

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


def test_dropped_worker_dies_with_its_last_reference(tmp_path):
    """A worker's captured graphs are in its ``_graphs``."""
    from llm_sharding_amd.config import get_preset
    from llm_sharding_amd.runtime.engine import RandomSource
    from llm_sharding_amd.utils.node_worker import NodeWorker
    cfg = get_preset("tiny")
    cfg.save_pretrained(str(tmp_path))
    w = NodeWorker("tcp://*:0", "tcp://127.0.0.1:1", False, str(tmp_path), dtype=torch.float32, backend="local", verbose=False,
                   max_seq=32, source=RandomSource(cfg, 0))
    w.load_shards(0, cfg.num_hidden_layers)
    assert w.past_key_value.get_seq_length() == 0
    w.engine.seq_len[0] = 5
    view = w.past_key_value
    assert view is w.past_key_value and view.get_seq_length() == 5
    gone = weakref.ref(w), weakref.ref(w.engine)
    gc.disable()
    try:
        del w
        assert [r() for r in gone] == [None, None] and view.get_seq_length() == 0
    finally:
        gc.enable()


@pytest.mark.parametrize("mode,split", [("first", True), ("mid", True), ("last", True), ("last", False)])
def test_recorded_handoffs_do_not_hold_their_graph(mode, split):
    """What a graph runs before and after its step sends the graph's buffers and leaves the graph to its owner."""
    from llm_sharding_amd.parallel.pipeline import PipelineStage
    said = []
    p2p = types.SimpleNamespace(recv=lambda t, r: said.append(("recv", t, r)), isend=lambda t, r: said.append(("send", t, r)))
    stage = types.SimpleNamespace(p2p=p2p, rank=2, mode=mode, split=split)
    g = _step(None)
    g.h_in, g._out = torch.zeros(1), torch.zeros(1)
    h_in, out, keys, tokens = g.h_in, g._out, g.keys, g.tokens
    PipelineStage._attach_comm(stage, g)
    if mode != "first":
        g.pre_comm()
    g.post_comm()
    want = [] if mode == "first" else [("recv", h_in, 1)]
    want += {"last": [("send", out, 0), ("send", keys, 0)] if split else [("send", tokens, 0)]}.get(mode, [("send", out, 3)])
    assert [(a, t.data_ptr(), r) for a, t, r in said] == [(a, t.data_ptr(), r) for a, t, r in want]
    gone = weakref.ref(g)
    gc.disable()
    try:
        del g
        assert gone() is None
    finally:
        gc.enable()
