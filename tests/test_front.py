"""The native half of the torch front end without a GPU: the records of a request, the fusion of a cycle, completion,
and what it hands back to Python."""
import ctypes
import os
import random
import sys
from decimal import Decimal
from fractions import Fraction

import pytest
import torch

from horovod_amd import _lib, build
from horovod_amd import workloads as W

F32, F16 = 7, 6


@pytest.fixture(scope="module")
def front():
    return _lib.front()


def _entry(front, name, n, dtype=torch.float32):
    t = torch.empty(n, dtype=dtype)
    return front.Entry(name, t, t)


def _request(front, entries, **kw):
    args = dict(op=1, prescale=1.0, postscale=0.5, tensor_dtype=F32, wire_dtype=F32, device=0)
    args.update(kw)
    return front.Request(entries, **args)


def _plan(front, requests, threshold, padded=True):
    fuse = ctypes.cast(_lib.adapter_lib().hvd_adapter_fuse_keyed, ctypes.c_void_p).value
    return front.plan(requests, padded, threshold, fuse)


@pytest.mark.parametrize("wire,es", [(F32, 4), (F16, 2)])
@pytest.mark.parametrize("padded", [True, False])
def test_a_cycle_fuses_by_bytes_on_the_wire(front, wire, es, padded):
    rng = random.Random(wire)
    counts = [rng.randrange(0, 3000) for _ in range(200)]
    requests = [_request(front, [_entry(front, str(i), c)], wire_dtype=wire) for i, c in enumerate(counts)]
    groups = _plan(front, requests, 20000, padded)
    want = W.fuse([c * es for c in counts], 20000, pad16=padded)
    assert [[int(e.name) for _, e in g] for g in groups] == want
    assert all(requests[int(e.name)] is r for g in groups for r, e in g)


def test_a_queue_is_emptied_into_the_list_that_is_taken(front):
    queue = [_request(front, [_entry(front, str(i), 1)]) for i in range(3)]
    want = list(queue)
    assert front.take(queue) == want and queue == [] and front.take(queue) == []
    with pytest.raises(TypeError):
        front.take(tuple(want))


def test_requests_of_different_kinds_do_not_share_a_response(front):
    variants = [{}, {"op": 2}, {"prescale": 0.25}, {"postscale": 1.0}, {"wire_dtype": F16}, {"tensor_dtype": 4, "wire_dtype": 4},
                {"device": 1}, {"kind": "allgather"}]
    requests = [_request(front, [_entry(front, "%d.%d" % (i, k), 10)], **v) for k in range(2) for i, v in enumerate(variants)]
    groups = _plan(front, requests, 1 << 20)
    assert sorted(sorted(e.name for _, e in g) for g in groups) == [["%d.0" % i, "%d.1" % i] for i in range(len(variants))]
    grouped = _request(front, [_entry(front, str(i), 1000) for i in range(3)], grouped=True)
    groups = _plan(front, [grouped], 8192)
    assert [len(g) for g in groups] == [2, 1] and all(r is grouped for g in groups for r, _ in g)


def test_requests_and_streams_of_a_response_come_once_each(front):
    entries = [_entry(front, str(i), 4) for i in range(5)]
    a, b, c = _request(front, entries[:2]), _request(front, entries[2:4]), _request(front, entries[4:])
    a.producer, b.producer, c.producer = (0, 0, 1), (7, 0, 1), tuple([0, 0, 1])
    group = [(a, entries[0]), (b, entries[2]), (a, entries[1]), (c, entries[4]), (b, entries[3])]
    assert front.requests(group) == ([a, b, c], [(0, 0, 1), (7, 0, 1)])
    marker = front.Marker(None, None, 3, [])
    front.attach([a, b, c], marker)
    assert [r.markers for r in (a, b, c)] == [[marker]] * 3 and marker.refs == 3 and marker.done is False


def test_completion_waits_for_every_marker_and_releases_an_event_once(front):
    inflight, handles, released = {}, {}, []
    state = front.State(2, 1, inflight, [], handles, [0], [0], released.append)
    first, second = front.Marker(None, 1, 2, []), front.Marker(None, 2, 1, [])
    one, two = (_request(front, [_entry(front, n, 4)]) for n in "ab")
    many = _request(front, [_entry(front, n, 4) for n in "cd"], grouped=True)
    for h, r in enumerate((one, two, many)):
        handles[h] = r
        inflight.update((e.name, r) for e in r.entries)
    front.attach([one, two], first)
    front.attach([many], second)
    assert state.finish(0) is front.PENDING  # not submitted
    for r in (one, two, many):
        r.submitted = True
    assert state.finish(0) is front.PENDING and len(handles) == 3  # not waited for
    first.done = True
    assert state.finish(0) is one.entries[0].output and released == [] and sorted(inflight) == ["b", "c", "d"]
    assert state.finish(0) is front.PENDING  # unknown by now
    two.error = ValueError("no")
    assert state.finish(1) is front.PENDING  # Python raises it
    two.error = None
    assert state.finish(1) is two.entries[0].output and released == [first]
    second.done = True
    outputs = state.finish(2)
    assert type(outputs) is list and all(o is e.output for o, e in zip(outputs, many.entries))
    assert released == [first, second] and not inflight and not handles and many.markers == []
    with pytest.raises(TypeError):
        state.finish([])


def test_what_is_not_plain_goes_back_to_python(front):
    """No tensor of the host is; those of the device are told apart in test_gpu_front.py."""
    handles, queue = {}, []
    state = front.State(2, 1, {}, queue, handles, [0], [0], print)
    t = torch.zeros(4)

    class Sub(torch.Tensor):
        pass

    for tensor in (t, t.as_subclass(Sub), torch.zeros(4, device="meta"), None, t.to_sparse(), [t]):
        assert state.submit(tensor, tensor, "x", 1, 1.0, 1.0, None) is None
        assert state.submit_group([tensor], [tensor], "x", 1, 1.0, 1.0, None) is None
    assert state.submit_group([], [], "x", 1, 1.0, 1.0, None) is None
    assert not handles and not queue
    with pytest.raises(TypeError):
        state.submit(t)
    group = [(_request(front, [_entry(front, "x", 4)]), _entry(front, "x", 4))]
    with pytest.raises(ZeroDivisionError):
        front.addresses(group, 3, lambda rank, name, tensor: 1 // 0, print)
    with pytest.raises(KeyError):  # a peer that is no device tensor is looked at by the callback
        front.addresses(group, 3, lambda rank, name, tensor: tensor, lambda t, e: {}[e.name])
    inputs, outputs, counts, peers = front.addresses(group, 3, None, print)
    at = group[0][1].tensor.data_ptr()
    assert list(inputs) == [at] * 3 and list(outputs) == [at] and list(counts) == [4] and peers == []
    inputs, _, _, peers = front.addresses(group, 3, lambda rank, name, tensor: t, lambda p, e: 4096)
    assert list(inputs) == [at, 4096, 4096] and len(peers) == 2 and peers[0] is t
    for bad in ([], [1], [(1, 2)]):
        with pytest.raises(TypeError):
            front.addresses(bad, 1, None, print)


def test_a_module_built_for_another_torch_or_interpreter_is_not_imported(front, monkeypatch, tmp_path):
    here = _lib.front_for()
    assert here.startswith(torch.__version__ + ",") and "cpython-%d%d" % sys.version_info[:2] in here
    monkeypatch.setattr(_lib, "_front", None)
    monkeypatch.setattr(_lib, "front_for", lambda: "2.0.0,other,cpython-30")
    with pytest.raises(RuntimeError, match="not built for this torch and interpreter"):
        _lib.front()
    monkeypatch.undo()
    monkeypatch.setattr(_lib, "_front", None)
    monkeypatch.setattr(_lib, "_HERE", str(tmp_path))
    os.mkdir(tmp_path / "lib")
    (tmp_path / "lib" / "_front.so").write_bytes(b"from before it said so")
    with pytest.raises(RuntimeError, match="not built for this torch and interpreter"):
        _lib.front()


def test_the_build_is_for_the_interpreter_that_asks(monkeypatch):
    commands = []
    monkeypatch.setattr(build.subprocess, "check_call", commands.append)
    build.build()
    assert "PYTHON=" + sys.executable in commands[0]


@pytest.mark.parametrize("factor", [0.5, 2, True, "0.25", Fraction(1, 8), Decimal("0.75"), torch.tensor(1.5), b"3"])
def test_a_factor_is_whatever_float_takes(front, factor):
    r = _request(front, [_entry(front, "a", 1)], prescale=factor, postscale=factor)
    assert r.prescale == r.postscale == float(factor)


@pytest.mark.parametrize("factor, error", [(None, TypeError), ("half", ValueError), (10 ** 400, OverflowError)])
def test_what_float_refuses_is_no_factor(front, factor, error):
    for which in ("prescale", "postscale"):
        with pytest.raises(error):
            _request(front, [_entry(front, "a", 1)], **{which: factor})
