"""A HIP graph that dies while another one is recorded ends the process: its destructor waits for the device, which a recording thread may
not do.  Graphs therefore go with the last reference to their engine, not in a cyclic collection, and none of those runs inside a
recording.  Without a GPU: the recording is a stand-in."""
import gc
import threading
import weakref

import pytest
import torch

from omniserve_amd import persistent
from omniserve_amd.engine import Engine, SequenceInput, engine as engine_module
from tests.test_engine_cpu import Pages


class Slots:
    """engine.batch.DecodeSlots without its pinned buffer"""

    def __init__(self, builder, places, width):
        self.builder, self.batch = builder, None

    def fill(self, entries):
        self.batch = self.builder.build(entries)[0]


class Step:
    """persistent.GraphedStep that runs its function eagerly"""
    made = []

    def __init__(self, fn, device=None):
        self.fn = fn
        Step.made.append(weakref.ref(self))

    def capture(self):
        pass

    def run(self):
        self.fn()


@pytest.fixture
def collector_off():
    on = gc.isenabled()
    gc.collect()
    gc.disable()
    yield
    if on:
        gc.enable()


def test_graphs_go_with_their_engine(monkeypatch, collector_off):
    monkeypatch.setattr(engine_module, "DecodeSlots", Slots)
    monkeypatch.setattr(engine_module, "GraphedStep", Step)
    Step.made.clear()
    engine = Engine(Pages(), max_tokens=1024)
    engine.use_graphs = True
    seq = engine.open()
    for t in (3, 5, 7):
        logits = engine.run([SequenceInput(seq, [t], [0])])
    plain = Engine(Pages(), max_tokens=1024)
    plain.use_graphs = False
    other = plain.open()
    for t in (3, 5, 7):
        want = plain.run([SequenceInput(other, [t], [0])])
    assert torch.equal(logits, want)
    assert len(Step.made) == 1 and Step.made[0]() is not None
    gone = weakref.ref(engine)
    del engine
    assert gone() is None and Step.made[0]() is None


class Loop:
    """only a cyclic collection takes it away"""

    def __init__(self):
        self.me = self


class Recording:
    """torch.cuda.graph's place"""

    def __init__(self, graph, **options):
        self.graph = graph

    def __enter__(self):
        self.graph.append("begin")

    def __exit__(self, *exc):
        self.graph.append("end")


def litter():
    """enough containers for collections of every generation"""
    return [[i] for i in range(400000)]


@pytest.fixture
def recording(monkeypatch):
    monkeypatch.setattr(torch.cuda, "graph", Recording)
    on = gc.isenabled()
    gc.enable()
    yield
    (gc.enable if on else gc.disable)()


def test_no_collection_inside_a_recording(recording):
    died = []

    def step():
        weakref.finalize(Loop(), died.append, 1)
        litter()
        assert not died and not gc.isenabled()

    graph = []
    persistent.record(graph, step)
    assert graph == ["begin", "end"] and gc.isenabled()
    litter()
    gc.collect()
    assert died


@pytest.mark.parametrize("on", [True, False])
def test_the_collector_is_left_as_it_was(recording, on):
    (gc.enable if on else gc.disable)()

    def failing():
        raise RuntimeError("in the step")

    with pytest.raises(RuntimeError, match="in the step"):
        persistent.record([], failing)
    assert gc.isenabled() == on
    persistent.record([], lambda: persistent.record([], lambda: None))
    assert gc.isenabled() == on


def test_recordings_of_two_threads(recording):
    """the first one that ends does not let the collector into the other one"""
    first, second, ended = threading.Event(), threading.Event(), threading.Event()
    states = []

    def one():
        first.set()
        assert second.wait(20)

    def two():
        second.set()
        assert ended.wait(20)
        states.append(gc.isenabled())

    a = threading.Thread(target=lambda: (persistent.record([], one), ended.set()))
    b = threading.Thread(target=lambda: (first.wait(20), persistent.record([], two)))
    a.start(), b.start()
    a.join(30), b.join(30)
    assert states == [False] and gc.isenabled()
