"""Stream ordering of a buffer's dispatches, on a model of streams and events that
remembers what every operation comes after (no GPU): whichever streams the dispatches of
one buffer run on, each comes after the one before (they share the ticket queues), after
its inputs and after every stream that consumed a result, and a synchronous one is in
front of what its caller's stream does next.  A synchronous one runs on the caller's stream
only where that may use every compute unit."""

from __future__ import annotations

import itertools
import random
import threading
from types import SimpleNamespace

import pytest

from pcie_ep import buffer as buffer_module
from pcie_ep.buffer import _Ordering
from pcie_ep.overlap import EventOverlap


class FakeGpu:
    """Streams hold the set of operations that are in front of whatever is put on them next."""

    def __init__(self, rng):
        self.handles, self.operations, self.rng = itertools.count(16), itertools.count(), rng
        self.finished, self.current = set(), None

        gpu = self

        class Stream:
            def __init__(self, device=None):
                self.device, self.cuda_stream, self.front = SimpleNamespace(index=0), next(gpu.handles), set()
                self.units = b"\xff"

            def put(self):
                operation = next(gpu.operations)
                before, self.front = self.front | gpu.finished, self.front | {operation}
                return operation, before

            def wait_event(self, event):
                self.front = self.front | event.front

            def wait_stream(self, other):
                self.front = self.front | other.front

            def query(self):
                if gpu.rng.random() < 0.5:  # everything on it has run
                    gpu.finished |= self.front
                return self.front <= gpu.finished

        class Event:
            front = frozenset()

            def record(self, stream):
                self.front = frozenset(stream.front)

        class Current:
            def __init__(self, stream):
                self.stream = stream

            def __enter__(self):
                self.before, gpu.current = gpu.current, self.stream

            def __exit__(self, *exc_info):
                gpu.current = self.before

        self.Stream, self.Event, self.Current = Stream, Event, Current


class Launched(Exception):
    pass


@pytest.fixture
def model(monkeypatch):
    def start(rng):
        gpu = FakeGpu(rng)
        cuda = SimpleNamespace(Stream=gpu.Stream, Event=gpu.Event, stream=gpu.Current, current_stream=lambda device=None: gpu.current)
        monkeypatch.setattr(buffer_module, "torch", SimpleNamespace(cuda=cuda))
        monkeypatch.setattr(buffer_module, "unit_mask", lambda stream: stream.units)
        gpu.current = gpu.Stream()
        return gpu

    return start


def test_a_thread_that_asks_for_the_stream_waits_for_the_dispatch_being_placed(model):
    gpu = model(random.Random(0))
    ordering = _Ordering(0)
    seen = []
    asking = threading.Thread(target=lambda: seen.append(ordering.expose().put()[1]))

    def work(stream):
        operation, _ = stream.put()
        asking.start()
        asking.join(0.1)  # it can not have been handed out: this dispatch has no completion event yet
        assert not seen
        return operation

    operation, _, _ = ordering.submit(work, synchronous=True)
    asking.join()
    assert operation in seen[0]
    place = []
    ordering.submit(place.append, synchronous=True)
    assert place == [ordering.stream]


@pytest.mark.parametrize("seed", range(6))
def test_every_dispatch_comes_after_the_one_before(model, seed):
    rng = random.Random(seed)
    for _ in range(50):
        walk(model(rng))


def walk(gpu):
    ordering = _Ordering(0)
    callers = [gpu.current] + [gpu.Stream() for _ in range(3)]
    few_units, unknown_units, default = callers[1:]
    few_units.units, unknown_units.units = b"\x0f", None
    default.units, default.cuda_stream = None, 0
    dispatches, exposed = [], False
    for _ in range(8):
        gpu.current = caller = gpu.rng.choice(callers)
        step = gpu.rng.choice(["synchronous", "synchronous", "asynchronous", "previous_event", "raises", "raises_async", "expose"])
        if step == "expose":
            stream = ordering.expose()
            _, before = stream.put()
            assert set(dispatches) <= before
            exposed = True
            continue
        produced, _ = caller.put()
        required = set(dispatches) | {produced}
        event = None
        if step == "previous_event":
            side = gpu.Stream()
            required = set(dispatches) | {side.put()[0]}
            event = EventOverlap(gpu.Event())
            event.event.record(side)
        # Results handed out so far are read by any of the streams, which say so.
        if dispatches and gpu.rng.random() < 0.5:
            consumer = gpu.rng.choice(callers)
            consumer.wait_event(ordering._last[1])
            required.add(consumer.put()[0])
            ordering.saw_consumer(consumer)
        synchronous = step in ("synchronous", "raises")
        place = []

        def work(stream):
            operation, before = stream.put()
            place.append(stream)
            dispatches.append(operation)
            assert required <= before, f"{step}: missing {required - before}"
            if step.startswith("raises"):
                raise Launched

        try:
            _, done, _ = ordering.submit(work, event, gpu.rng.random() < 0.5, synchronous)
        except Launched:
            pass
        else:
            assert dispatches[-1] in done.front
            if synchronous:
                assert dispatches[-1] in caller.put()[1]
                ordering.saw_consumer(caller)
        assert gpu.current is caller
        holds = caller is default or caller.units == b"\xff"
        in_line = synchronous and not exposed and holds
        assert place[0] is (caller if in_line else ordering.stream)
