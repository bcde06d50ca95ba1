"""The queue and the cycles of the torch engine without a GPU: its streams and what a response does are stand-ins."""
import sys
import threading
import time

import pytest
import torch

from horovod_amd.torch import engine

F32 = 7


class _Stream:
    handle = None

    def destroy(self):
        pass


@pytest.fixture
def make_engine(monkeypatch):
    monkeypatch.setattr(engine.H, "Stream", _Stream)
    monkeypatch.setattr(engine, "_current_stream", lambda: (0, 0, 1))

    def make(execute, **kw):
        """An engine whose responses are `execute(group)`."""
        monkeypatch.setattr(engine.Engine, "_execute", lambda self, group: execute(group))
        monkeypatch.setattr(engine.Engine, "_release", lambda self, marker: None)
        return engine.Engine(**kw)

    interval = sys.getswitchinterval()
    yield make
    sys.setswitchinterval(interval)


_T = torch.empty(4)


def _complete(group):
    """What a response that has completed leaves with its requests."""
    requests, _ = engine._front.requests(group)
    marker = engine.Marker(None, None, len(requests), [])
    marker.done = True
    engine._front.attach(requests, marker)


def _request(*names):
    return engine.Request([engine.Entry(n, _T, _T) for n in names], engine.SUM, 1.0, 1.0, F32, F32, 0, grouped=len(names) > 1)


def test_no_request_is_lost_between_threads(make_engine):
    """One thread enqueues while another runs cycles, as a thread that averages a metric does beside the one that waits for
    gradients: every request goes through one response."""
    seen = []
    eng = make_engine(lambda group: seen.extend(e.name for _, e in group))
    count, done = 20000, threading.Event()
    sys.setswitchinterval(1e-5)

    def enqueue():
        try:
            for i in range(count):
                eng.enqueue(_request(str(i)))
        finally:
            done.set()

    thread = threading.Thread(target=enqueue)
    thread.start()
    while not done.is_set():
        eng.run_cycle()
    thread.join()
    eng.run_cycle()
    assert seen == [str(i) for i in range(count)]
    assert all(r.submitted for r in eng.inflight.values())


def test_cycles_of_two_threads_do_not_overlap(make_engine):
    """They share the stream slots, and with them buffers that several launches of a response go through."""
    inside, overlapped, completed = [0], [], []

    def execute(group):
        inside[0] += 1
        if inside[0] > 1:
            overlapped.append([e.name for _, e in group])
        time.sleep(1e-4)  # where launches let other threads run
        inside[0] -= 1
        completed.extend(e.name for _, e in group)
        _complete(group)

    eng = make_engine(execute)
    missed = []

    def work(which):
        for i in range(200):
            r = _request("%s%d" % (which, i))
            eng.enqueue(r)
            eng.wait(r)
            if r.entries[0].name not in completed:
                missed.append(r.entries[0].name)

    threads = [threading.Thread(target=work, args=(w,)) for w in "abc"]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not overlapped and not missed and not eng.inflight and len(completed) == 600


def test_a_request_of_another_threads_cycle_is_waited_for(make_engine):
    started, go_on = threading.Event(), threading.Event()

    def execute(group):
        started.set()
        assert go_on.wait(30)
        _complete(group)

    eng = make_engine(execute)
    r, done = _request("a"), []
    eng.enqueue(r)
    cycle = threading.Thread(target=eng.run_cycle)
    cycle.start()
    assert started.wait(30)
    waiting = threading.Thread(target=lambda: (eng.wait(r), done.append(True)))
    waiting.start()
    waiting.join(0.2)
    assert waiting.is_alive() and not done
    assert eng.poll(r) is False  # and does not wait
    go_on.set()
    cycle.join()
    waiting.join()
    assert done and r.submitted and not eng.inflight


def test_within_a_cycle_only_what_has_been_executed_can_be_waited_for(make_engine):
    """As a peer_source might: of its own response, or a later one, there is nothing to wait for yet."""
    said = []

    def execute(group):
        for r in requests:
            try:
                eng.wait(r)
                said.append("done")
            except engine.HorovodInternalError as e:
                said.append(str(e))
            if "its own cycle" in said[-1]:
                assert eng.poll(r) is False
        if group[0][1].name == "b":
            raise ValueError("no")
        _complete(group)

    eng = make_engine(execute, fusion_threshold=0)
    requests = [_request("a"), _request("b"), _request("c", "d")]
    for r in requests:
        eng.enqueue(r)
    eng.run_cycle()
    early = "An operation cannot be waited for from within its own cycle before its response."
    assert said == [early] * 3 + ["done", early, early] + ["done", "no", early] * 2
    eng.wait(requests[2])
    assert not eng.inflight


def test_what_an_interrupted_cycle_left_out_is_an_error(make_engine):
    class Interrupt(BaseException):
        pass

    def execute(group):
        if group[0][1].name != "a":
            raise Interrupt("stop")
        _complete(group)

    eng = make_engine(execute, fusion_threshold=0)
    requests = [_request(n) for n in "abc"]
    for r in requests:
        eng.enqueue(r)
    with pytest.raises(Interrupt):
        eng.run_cycle()
    eng.wait(requests[0])
    for r in requests[1:]:
        with pytest.raises(engine.HorovodInternalError, match="stop"):
            eng.wait(r)
    assert not eng.inflight
