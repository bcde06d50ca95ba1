"""The native half of the torch front end on the GPU: tensors and peers that are not the plain case take the Python path
and give the same, work of busy streams is waited for whether or not the engine looks, and nothing is left behind."""
import ctypes
import gc
import threading

import pytest
import torch

import horovod_amd
from horovod_amd._lib import check, front

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


@pytest.fixture
def hvd():
    import horovod_amd.torch as hvd
    hvd.shutdown()
    yield hvd
    hvd.shutdown()


KINDS = {"plain": lambda t: t, "parameter": lambda t: torch.nn.Parameter(t, requires_grad=False),
         "subclass": lambda t: t.as_subclass(Sub)}


@pytest.mark.parametrize("peer", KINDS)
@pytest.mark.parametrize("own", KINDS)
def test_every_kind_of_tensor_is_summed(hvd, own, peer):
    hvd.init(size=3, peer_source=lambda rank, name, t: KINDS[peer](torch.full_like(t.data, float(rank)).as_subclass(torch.Tensor)))
    t = KINDS[own](torch.arange(1000, dtype=torch.float32, device="cuda"))
    out = hvd.synchronize(hvd.allreduce_async(t, op=hvd.Sum))
    assert torch.equal(out.as_subclass(torch.Tensor), t.as_subclass(torch.Tensor) + 3)
    rows = hvd.synchronize(hvd.allgather_async(t.reshape(10, 100), name="rows"))
    assert rows.shape == (30, 100) and torch.equal(rows.as_subclass(torch.Tensor)[10:], torch.cat(
        [torch.full((10, 100), float(r), device="cuda") for r in (1, 2)]))


def test_what_is_not_the_plain_case_is_not_submitted_natively():
    """Whatever the native half hands back reaches the checks in Python; it leaves nothing behind then."""
    handles, queue, inflight, next_handle, noname = {}, [], {}, [0], [0]
    state = front().State(6, 2, inflight, queue, handles, next_handle, noname, print)
    t = torch.zeros(4, 6, device="cuda")
    plain = dict(tensor=t, output=torch.zeros_like(t), name=None, op=1, pre=1.0, post=1.0, wire=None)

    def submitted(**changed):
        a = {**plain, **changed}
        rest = (a["op"], a["pre"], a["post"], a["wire"])
        one = state.submit(a["tensor"], a["output"], a["name"], *rest)
        group = state.submit_group([t, a["tensor"]], [t, a["output"]], str(a["name"]), *rest)
        return one, group

    wrapped = []

    def inside(x):
        wrapped.append(submitted(tensor=x, output=x))
        return x.sum()

    torch.func.vmap(inside)(t)
    torch.func.grad(inside)(t)
    functional = torch._to_functional_tensor(t)
    nested = torch.nested.nested_tensor([t[0], t[1]])
    refused = [submitted(tensor=x, output=x) for x in (
        t.as_subclass(Sub), t.to_sparse(), t.t(), t[:, ::2], functional, nested, t.cpu(), t.to(torch.bfloat16), None)]
    refused += [submitted(output=x) for x in (
        torch.zeros(6, 4, device="cuda"), t.double(), t.cpu(), torch.zeros(6, 4, device="cuda").t(), t.as_subclass(Sub), None)]
    refused += [submitted(op=x) for x in (3, -1, 1 << 70, True, 1.0, None, 2)]  # Adasum of three nodes, too
    refused += [submitted(**{k: x}) for k in ("pre", "post") for x in (True, 1 << 60, "1", None, torch.tensor(1.0))]
    refused += [submitted(wire=x) for x in (torch.bfloat16, "fp16", 6)]
    assert len(wrapped) == 2 and all(r == (None, None) for r in wrapped + refused), refused
    assert state.submit(t, t, 7, 1, 1.0, 1.0, None) is None
    assert state.submit_group([t, t.double()], [t, t], "x", 1, 1.0, 1.0, None) is None
    assert state.submit_group([t], [t, t], "x", 1, 1.0, 1.0, None) is None
    assert not handles and not queue and not inflight and next_handle == noname == [0]
    for i, changed in enumerate((dict(name="x"), dict(output=t), dict(op=0, pre=2, wire=torch.float16),
                                 dict(tensor=torch.nn.Parameter(t), name="y"))):
        assert submitted(**changed) == (2 * i + 1, 2 * i + 2)
        assert submitted(**{**plain, "name": "x"}) == (None, None)  # in flight
        inflight.pop("None_1of2", None), inflight.pop("None_2of2", None)
    assert sorted(handles) == list(range(1, 9)) and queue == list(handles.values()) and noname == [2]


@pytest.mark.parametrize("odd", [None, 0, 1, 2])
def test_a_group_is_summed_whatever_its_tensors_are(hvd, odd):
    """One that is no plain tensor takes the whole group through Python; the names and results are the same."""
    names = []

    def source(rank, name, t):
        names.append(name)
        return torch.full_like(t, float(rank))

    hvd.init(size=2, peer_source=source)
    tensors = [torch.arange(n, dtype=torch.float32, device="cuda") for n in (5, 1000, 1)]
    if odd is not None:
        tensors[odd] = tensors[odd].as_subclass(Sub)
    for out, t in zip(hvd.synchronize(hvd.grouped_allreduce_async(tensors, name="g", op=hvd.Sum)), tensors):
        assert torch.equal(out.as_subclass(torch.Tensor), t.as_subclass(torch.Tensor) + 1)
    assert names == ["grouped_allreduce.g_%dof3" % i for i in (1, 2, 3)]
    first = hvd.grouped_allreduce_async(tensors, name="g")
    with pytest.raises(hvd.HorovodInternalError, match="same name"):
        hvd.grouped_allreduce_async(tensors, name="g")
    hvd.synchronize(first)
    with pytest.raises(ValueError, match="share dtype and device"):
        hvd.grouped_allreduce_async([tensors[0], tensors[1].double()])


def test_an_unnamed_tensor_does_not_take_a_name_in_flight(hvd):
    """Unnamed tensors are numbered; one that a script has named like the next of them is in its way until it is finished."""
    from horovod_amd.torch import mpi_ops
    hvd.init(size=2)
    for kind in (KINDS["plain"], KINDS["subclass"]):  # both ways in
        t = kind(torch.arange(100, dtype=torch.float32, device="cuda"))
        taken = hvd.allreduce_async(t, name="noname.%d" % (mpi_ops._noname[0] + 1), op=hvd.Sum)
        with pytest.raises(hvd.HorovodInternalError, match="same name"):
            hvd.allreduce_async(t, op=hvd.Sum)
        assert len(mpi_ops._engine.inflight) == 1
        later = hvd.allreduce_async(t, op=hvd.Sum)  # the next number
        for h in (later, taken):
            assert torch.equal(hvd.synchronize(h).as_subclass(torch.Tensor), 2 * t.as_subclass(torch.Tensor))
        assert not mpi_ops._engine.inflight


@pytest.mark.parametrize("wrong", [lambda t: t.double(), lambda t: t[:-1], lambda t: t.cpu(), lambda t: None,
                                   lambda t: torch.stack([t, t], 1)[:, 0], lambda t: t.double().as_subclass(Sub)])
def test_a_peer_that_does_not_fit_is_an_error_of_its_response(hvd, wrong):
    hvd.init(size=2, peer_source=lambda rank, name, t: wrong(t) if name.endswith("bad") else t)
    t = torch.ones(100, device="cuda")
    handle = hvd.allreduce_async(t, name="bad")
    with pytest.raises(hvd.HorovodInternalError, match="peer_source must return"):
        hvd.synchronize(handle)
    assert torch.equal(hvd.allreduce(t, name="good"), t)


@pytest.mark.parametrize("peers", [True, False])
@pytest.mark.parametrize("stream", ["default", "side", "another than at the cycle"])
def test_work_of_a_busy_stream_is_waited_for(hvd, stream, peers):
    """The tensor (and in turn the peer's) is written behind a long wait on the device: in cycles in which the engine looks
    at the stream and finds it busy, in those after, in which it does not look, and among idle ones."""
    y = torch.zeros(1 << 16, device="cuda")
    hvd.init(size=2, peer_source=(lambda rank, name, t: y) if peers else None)
    other = torch.cuda.current_stream() if stream == "default" else torch.cuda.Stream()
    x = torch.zeros(1 << 16, device="cuda")
    torch.cuda.synchronize()
    for i in range(40):
        with torch.cuda.stream(other):
            if i % 20 < 4 or i % 3 == 0:
                torch.cuda._sleep(2000000)
            x.fill_(i)
            y.fill_(2 * i if peers else i)
            handle = hvd.allreduce_async(x, op=hvd.Sum)
            if stream != "another than at the cycle":
                out = hvd.synchronize(handle)
        if stream == "another than at the cycle":
            if peers:  # they are made on the stream of the cycle, which here waits for the other
                torch.cuda.current_stream().wait_stream(other)
            out = hvd.synchronize(handle)
        assert float(out[0]) == float(out[-1]) == (3 * i if peers else 2 * i), i
        other.synchronize()


@pytest.mark.parametrize("n", [1, 1000, 1 << 20, 5 << 20])
def test_what_an_idle_stream_has_written_is_read(hvd, n):
    """Without an event between the two streams: tensors that the sum has read before, so that its caches may hold them,
    rewritten on the framework's stream, which is then only polled until it has nothing left."""
    x, y = (torch.zeros(n, device="cuda") for _ in range(2))
    hvd.init(size=3, peer_source=lambda rank, name, t: y)
    out = torch.empty_like(x)
    stream = torch.cuda.current_stream()
    for i in range(200):
        x.fill_(i)
        y.fill_(3 * i)
        while not stream.query():
            pass
        out = hvd.synchronize(hvd.allreduce_async(x, name="t", op=hvd.Sum))
        assert float(out.min()) == float(out.max()) == 7 * i, i


def test_idle_is_said_of_idle_streams_only():
    L = horovod_amd.lib()

    def idle(s):
        out = ctypes.c_int(-1)
        check(L.hvdhip_stream_idle(s.cuda_stream, ctypes.byref(out)), "hvdhip_stream_idle")
        return out.value

    for s in (torch.cuda.default_stream(), torch.cuda.Stream()):
        torch.cuda.synchronize()
        assert idle(s) == 1
        with torch.cuda.stream(s):
            torch.cuda._sleep(20000000)
        assert idle(s) == 0
        assert float((torch.ones(8, device="cuda") + 1)[0]) == 2.0  # no stale error is left for the next launch
        s.synchronize()
        assert idle(s) == 1
    assert L.hvdhip_stream_idle(None, None) == -1
    x, g, s = torch.zeros(64, device="cuda"), torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        x.add_(1)
        assert idle(s) == 0  # and the capture goes on
        x.add_(1)
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert float(x[0]) == 2 * (i + 1)


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("stream", ["default", "side"])
@pytest.mark.parametrize("where", ["here", "in another thread"])
def test_the_capture_of_another_stream_goes_on(hvd, where, stream, mode):
    """Whoever asks for a stream that is not being captured, or hands over and waits for a tensor there in another thread, is
    no concern of a capture that is going on."""
    L = horovod_amd.lib()
    hvd.init(size=2)
    cur = torch.cuda.default_stream() if stream == "default" else torch.cuda.Stream()
    x, t = torch.zeros(64, device="cuda"), torch.ones(64, device="cuda")
    g, said = torch.cuda.CUDAGraph(), []

    def work():
        try:
            with torch.cuda.stream(cur):
                for _ in range(3):
                    idle = ctypes.c_int(-1)
                    check(L.hvdhip_stream_idle(cur.cuda_stream, ctypes.byref(idle)), "hvdhip_stream_idle")
                    said.append(idle.value)
                    if where != "here":
                        hvd.synchronize(hvd.allreduce_async_(t, op=hvd.Sum))
        except Exception as e:
            said.append(repr(e))

    with torch.cuda.stream(cur):
        hvd.synchronize(hvd.allreduce_async_(t, op=hvd.Average))
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
        x.add_(1)
        if where == "here":
            work()
        else:
            thread = threading.Thread(target=work)
            thread.start()
            thread.join()
        x.add_(1)
    assert said == [1] * 3
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert float(x.sum()) == 64 * 2 * (i + 1)
    assert float(t.sum()) == (64 if where == "here" else 64 * 2 ** 3)


def test_the_stream_of_a_request_is_the_current_one(hvd, gpu):
    from horovod_amd.torch import engine, mpi_ops
    hvd.init(size=2)
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.ExternalStream(gpu.stream.handle.value)):
        with torch.cuda.stream(stream):
            assert mpi_ops._state_of_front.producer() == tuple(engine._current_stream())


def test_nothing_is_left_of_finished_requests(hvd):
    t = [torch.ones(1000, device="cuda") for _ in range(20)]
    hvd.init(size=4, peer_source=lambda rank, name, x: torch.ones_like(x))

    def step(i):
        handles = [hvd.allreduce_async(x, name="%d" % k if i % 2 else None) for k, x in enumerate(t)]
        for h in handles:
            hvd.synchronize(h)

    def counts():
        gc.collect()
        torch.cuda.synchronize()
        kinds = (front().Request, front().Entry, front().Marker)
        return torch.cuda.memory_allocated(), sum(type(o) in kinds for o in gc.get_objects())

    for i in range(4):
        step(i)
    before = counts()
    for i in range(50):
        step(i)
    assert counts() == before and before[1] == 0


def test_behind_a_large_response_a_cycle_keeps_its_stream(hvd, monkeypatch):
    from horovod_amd.torch import engine, mpi_ops
    hvd.init(size=2, num_streams=2, fusion_threshold=0)  # a response per tensor
    monkeypatch.setattr(engine, "_BYTES_OF_ITS_OWN", 2 * 4 * 1000)
    slots, begin = [], engine.Engine._begin

    def recorded(self, group, made=None, nbytes=0):
        found = begin(self, group, made, nbytes)
        slots.append(found[0])
        return found

    monkeypatch.setattr(engine.Engine, "_begin", recorded)
    for sizes in ((999, 999, 5), (4, 1000, 5, 4000, 1), (7,), (7,)):
        tensors = [torch.full((n,), 1.5, device="cuda") for n in sizes]
        handles = [hvd.allreduce_async(t, op=hvd.Sum) for t in tensors]
        for h, t in zip(handles, tensors):
            assert torch.equal(hvd.synchronize(h), 2 * t)
    assert slots == [0, 1, 0] + [1, 0, 0, 0, 0] + [0] + [1]


def test_threads_share_the_engine(hvd):
    """Two threads on streams of their own hand over and wait: Adasum of several ranks, whose levels go through a workspace
    of the stream slot, sums and allgathers.  Each gets what it gets alone, whichever thread's cycle executes it."""
    hvd.init(size=8, peer_source=lambda rank, name, t: t * (1 + rank % 3))
    torch.manual_seed(1)
    sets = [[torch.randn(n, device="cuda") for n in (300000, 5, 70001, 40000)] for _ in range(2)]

    def step(tensors, tag):
        handles = [hvd.grouped_allreduce_async(tensors, name=tag + "a", op=hvd.Adasum), hvd.allreduce_async(tensors[0], name=tag + "s"),
                   hvd.allgather_async(tensors[2], name=tag + "g")]
        adasum, total, rows = [hvd.synchronize(h) for h in reversed(handles)][::-1]
        return adasum + [total, rows]

    want = [step(tensors, "alone") for tensors in sets]
    torch.cuda.synchronize()
    wrong = []

    def work(which):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(60):
                    got = step(sets[which], "%d.%d" % (which, i))
                    wrong.extend((which, i, k) for k, (g, w) in enumerate(zip(got, want[which])) if not torch.equal(g, w))
        except Exception as e:
            wrong.append((which, repr(e)))

    threads = [threading.Thread(target=work, args=(w,)) for w in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("peers", [True, False])
def test_the_null_stream_is_busy_with_a_blocking_one(hvd, peers):
    """An event on the null stream lies behind all that blocking streams, as other libraries make them, hold by then.  The
    look at the null stream has to say the same, or a tensor written there is read too early."""
    L = horovod_amd.lib()
    handle, idle = ctypes.c_void_p(), ctypes.c_int(-1)
    assert L.hipStreamCreateWithFlags(ctypes.byref(handle), 0) == 0  # of the HIP runtime below the library
    other = torch.cuda.ExternalStream(handle.value)
    x, y = (torch.zeros(1 << 16, device="cuda") for _ in range(2))
    hvd.init(size=2, peer_source=(lambda rank, name, t: y) if peers else None)
    torch.cuda.synchronize()
    assert torch.cuda.current_stream().cuda_stream == 0
    for i in range(1, 21):
        with torch.cuda.stream(other):
            torch.cuda._sleep(2000000)
            x.fill_(i)
            y.fill_(2 * i)
        if i % 6 == 1:  # the engine looks, too: it takes a stream that it found busy to be so for four cycles
            check(L.hvdhip_stream_idle(None, ctypes.byref(idle)), "hvdhip_stream_idle")
            assert idle.value == 0
        out = hvd.synchronize(hvd.allreduce_async(x, op=hvd.Sum))
        assert float(out[0]) == float(out[-1]) == (3 * i if peers else 2 * i), i
        torch.cuda.synchronize()
    check(L.hvdhip_stream_idle(None, ctypes.byref(idle)), "hvdhip_stream_idle")
    assert idle.value == 1
    assert L.hipStreamDestroy(handle) == 0


@pytest.mark.parametrize("peers", [True, False])
@pytest.mark.parametrize("stream", ["default", "side"])
@pytest.mark.parametrize("behind", ["a wait for another stream", "a graph", "a graph of two branches", "a copy from the host"])
def test_a_stream_is_busy_with_whatever_it_holds(hvd, behind, stream, peers):
    """What a framework's stream has to do may be no kernel of its own: the look has to find it all the same."""
    x, y = (torch.zeros(1 << 16, device="cuda") for _ in range(2))
    hvd.init(size=2, peer_source=(lambda rank, name, t: y) if peers else None)
    cur = torch.cuda.default_stream() if stream == "default" else torch.cuda.Stream()
    other, host = torch.cuda.Stream(), torch.zeros(1 << 16).pin_memory()
    i_dev = torch.zeros(1, device="cuda")

    def write():
        torch.cuda._sleep(2000000)
        x.copy_(i_dev.expand_as(x))
        y.copy_((2 * i_dev).expand_as(y))

    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    if behind.startswith("a graph"):
        capturing = torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=capturing):
            if behind == "a graph":
                write()
            else:
                other.wait_stream(capturing)
                with torch.cuda.stream(other):
                    write()
                capturing.wait_stream(other)
    for i in range(1, 21):
        i_dev.fill_(i)
        torch.cuda.synchronize()
        with torch.cuda.stream(cur):
            if behind.startswith("a graph"):
                graph.replay()
            elif behind == "a wait for another stream":
                with torch.cuda.stream(other):
                    write()
                cur.wait_stream(other)
            else:
                torch.cuda._sleep(2000000)
                host.fill_(i)
                x.copy_(host, non_blocking=True)
                y.copy_(host, non_blocking=True)
            out = hvd.synchronize(hvd.allreduce_async(x, op=hvd.Sum))
        want = i + (i if not peers or behind == "a copy from the host" else 2 * i)
        assert float(out.min()) == float(out.max()) == want, i
        torch.cuda.synchronize()
