"""The queue and the cycles of the torch engine without a GPU: its streams and what a response does are stand-ins."""
import sys
import threading

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
        return engine.Engine(**kw)

    interval = sys.getswitchinterval()
    yield make
    sys.setswitchinterval(interval)


_T = torch.empty(4)


def _request(name):
    return engine.Request([engine.Entry(name, _T, _T)], engine.SUM, 1.0, 1.0, F32, F32, 0)


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
