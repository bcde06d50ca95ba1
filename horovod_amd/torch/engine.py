"""What sits between ``allreduce_async_()`` and the kernels, for one process and one GPU.

In the reference a background thread negotiates which tensors are ready on every rank,
fuses the responses (Controller::FuseResponses, common/controller.cc:793-866) and runs the
allreduce op on each fused response (NCCLAllreduce::Execute, ops/nccl_operations.cc:156-214;
AdasumGpuAllreduceOp, ops/adasum_gpu_operations.cc:64-310).  Here there is nothing to
negotiate: a cycle takes every request enqueued since the last one, fuses them with the same
rule (through the C++ adapter) and queues, for every fused response,

    wait for the framework's ready events -> the sum over ranks in one pass (prescale, optional fp16
    narrowing, the additions in rank order, postscale, widening) -> completion event

on one of the engine's streams through the C ABI of libhvdhip.so.  Nothing here computes.

One GPU cannot hold a real communicator, so the *world* is simulated: ``size`` ranks of which
this process is rank 0.  What ranks 1..size-1 contribute comes from ``peer_source(rank, name,
tensor)``; by default every rank holds the same values, which is what the reference's own
tests arrange by seeding all ranks alike (test/parallel/test_torch.py:251-445).  All of
them sit in this GPU's memory, so a sum needs no fusion buffer: the kernel reads every rank's tensors
where they are, with the roundings that packing, summing and unpacking would make.  Adasum reads them
so too, a pass per level of the pairwise tree; only where a node has several ranks are these summed into
a buffer per node first.
"""
import ctypes
import threading
from ctypes import c_int, c_void_p

import torch

from .. import host as H
from .._lib import adapter_lib, check, dtype_size, front, lib

SUM = 1      # ReduceOp values, common/operations.h:35-40
ADASUM = 2

TORCH_TO_HVD = {
    torch.uint8: 0, torch.int8: 1, torch.int16: 3, torch.int32: 4, torch.int64: 5,
    torch.float16: 6, torch.float32: 7, torch.float64: 8, torch.bool: 9,
}
_ADASUM_DTYPES = (6, 7, 8)


def _current_stream():
    """What torch.cuda.current_stream() makes its Stream object from: (stream_id, device_index, device_type).  One per
    tensor is enough of them to matter (2.5 us for the object, 0.3 us for this)."""
    return torch._C._cuda_getCurrentStream(torch._C._cuda_getDevice())


def _stream_of(producer):
    stream_id, device_index, device_type = producer
    return torch.cuda.Stream(stream_id=stream_id, device_index=device_index, device_type=device_type)


class HorovodInternalError(RuntimeError):
    """An error of the op layer surfacing in the caller (horovod/common/exceptions.py:18-23)."""


# The records that travel through a cycle, and the loops over tensors and ranks, are native (csrc/front/front.cc):
#   Entry(name, tensor, output)        count = elements; parts = what every rank contributes to an allgather
#   Request(entries, op, prescale, postscale, tensor_dtype, wire_dtype, device, kind, grouped)
#       producer = the framework stream that was current at enqueue (torch's identifiers); markers = one Marker per
#       fused response that carries one of the entries; submitted, error
#   Marker(stream, event, refs, keepalive)   completion event of one fused response, shared by the requests it carried
#       (ops/gpu_operations.cc:50-56 records one per response); done; keepalive = the other ranks' tensors until then
_front = front()
Entry, Request, Marker = _front.Entry, _front.Request, _front.Marker


def _is_peer(t, tensor, count):
    """Whether t can stand for another rank's `tensor`: for those that the native check leaves open."""
    return (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == tensor.dtype and t.numel() == count
            and t.is_contiguous())


def _peer_address(t, e):
    if not _is_peer(t, e.tensor, e.count):
        raise ValueError("peer_source must return a contiguous device tensor of the shape and dtype of %r" % e.name)
    return t.data_ptr()


def _is_part(t, e):
    """Whether t can stand for another rank's rows of an allgather (first dimensions may differ)."""
    return (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == e.tensor.dtype and t.dim() == e.tensor.dim()
            and t.shape[1:] == e.tensor.shape[1:] and t.is_contiguous())


# Behind a response that reads this many bytes, all ranks together, the others of its cycle stay on its stream: each has
# the memory to itself then, where two at a time stream 3 to 5 % slower between them and the first completes with the second.
# Below, the start and the end of a response hide in the other's work.  Four responses on one stream and on two, us: 8
# ranks, 256 MB each 199 and 197, 320 MB 241 and 242, 512 MB 367 and 371, 1,280 MB 890 and 920; 2 ranks, 128 MB 141 and
# 133, 320 MB 314 and 316, 960 MB 882 and 911; 16 ranks, 320 MB 242 and 250.
_BYTES_OF_ITS_OWN = 320 << 20

# Cycles for which a framework stream that was found busy is waited for without another look.  A look costs 0.1 us at an
# idle stream and saves the event and the wait, 15 us of host time for every response; at a busy one it costs 6 to 8 us on
# top of them.  Few, so that a script whose stream is idle again soon has what the look saves, and more than none for one
# that averages a value it has just computed.
_BUSY_CYCLES = 4


class Engine:
    def __init__(self, size=1, local_size=1, peer_source=None, fusion_threshold=64 << 20, num_streams=1,
                 batch_d2d_memcopies=True):
        if size < 1 or local_size < 1 or size % local_size:
            raise ValueError("size must be a positive multiple of local_size")
        self.size, self.local_size, self.peer_source = size, local_size, peer_source
        self.fusion_threshold = int(fusion_threshold)
        self.batch_d2d_memcopies = bool(batch_d2d_memcopies)
        self.streams = [H.Stream() for _ in range(max(1, num_streams))]
        self.slot = 0
        # Held for a whole cycle: the slots, their buffers and events are one thread's at a time, and whoever waits for a
        # request that another thread's cycle has taken waits for that cycle first.  Again by the same thread where
        # peer_source calls back.
        self.cycling = threading.RLock()
        self.queue = []
        self.inflight = {}       # tensor name -> request, until synchronised
        self.buffers = {}        # (slot, what for) -> torch uint8 tensor
        self.cycles = 0
        self.responses = 0       # fused responses executed so far
        self.ready = {}          # framework stream -> event recorded during the current cycle
        self.staying = 0         # the last cycle with a response whose stream the others behind it keep to
        self.busy = {}           # framework stream -> cycle up to which it is taken to be busy

    # ---- queueing -------------------------------------------------------

    def enqueue(self, request):
        inflight = self.inflight
        for e in request.entries:
            if e.name in inflight:
                # common/tensor_queue.cc:27-31
                raise HorovodInternalError(
                    "Requested to allreduce a tensor with the same name as another tensor that is "
                    "currently being processed.  If you want to request another tensor, use a different "
                    "tensor name.")
        for e in request.entries:
            inflight[e.name] = request
        # The reference records a ready event per request on the framework's stream
        # (RecordReadyEvent, horovod/torch/ready_event.cc).  A cycle here runs on the caller's own
        # thread, after every enqueue it serves, so one event per producing stream and cycle, recorded
        # during the cycle, orders the same work and costs one record instead of one per tensor.
        if request.kind == "allgather":
            self._prepare_allgather(request)
        request.producer = _current_stream()
        self.queue.append(request)

    def _prepare_allgather(self, request):
        """Collects what every rank passes (first dimensions may differ, the rest may not:
        AllgatherOp::AllocateOutput, ops/collective_operations.cc:150-198) and allocates the
        output, here, before the cycle's ready event, so that its memory is ordered like any
        other tensor of the framework."""
        for e in request.entries:
            if e.tensor.dim() == 0:
                self.inflight.pop(e.name, None)
                # common/controller.cc:575-579
                raise HorovodInternalError("Rank zero tried to allgather a rank-zero tensor.")
            found = _front.parts(e, self.size, self.peer_source, _is_part)
            if found is None:
                self.inflight.pop(e.name, None)
                raise HorovodInternalError(
                    "Mismatched allgather tensor shapes: ranks may differ in the first dimension only "
                    "(tensor %r)." % e.name)
            e.parts, rows = found
            e.output.resize_((rows,) + tuple(e.tensor.shape[1:]))

    def run_cycle(self):
        """Fuses and queues everything enqueued so far (one pass of RunLoopOnce,
        common/operations.cc:593-717, with every request already agreed upon)."""
        with self.cycling:
            pending = _front.take(self.queue)  # other threads may be enqueuing
            if not pending:
                return
            self.cycles += 1
            self.ready = {}
            try:
                fuse = ctypes.cast(adapter_lib().hvd_adapter_fuse_keyed, c_void_p).value
                for g in _front.plan(pending, self.batch_d2d_memcopies, self.fusion_threshold, fuse):
                    try:
                        if g[0][0].kind == "allgather":
                            self._execute_allgather(g)
                        else:
                            self._execute(g)
                    except Exception as exc:  # surfaces in synchronize(), like a Status passed to the callback
                        for r, _ in g:
                            r.error = exc
                    _front.executed(g)
            except BaseException as exc:  # an interrupt: the rest is not executed
                for r in pending:
                    if not r.submitted:
                        r.error, r.submitted = exc, True
                raise

    # ---- resources ------------------------------------------------------

    def _buffer(self, slot, what, nbytes):
        t = self.buffers.get((slot, what))
        if t is None or t.numel() < nbytes:
            if t is not None:
                self.streams[slot].synchronize()  # queued kernels may still use the smaller buffer
            t = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")
            self.buffers[(slot, what)] = t
        return t.data_ptr()

    # ---- one fused response --------------------------------------------

    def _execute(self, group):
        first = group[0][0]
        # rank-major: inputs[rank * len(group) + entry]
        inputs, outputs, counts, peers = _front.addresses(group, self.size, self.peer_source, _peer_address)
        # the other ranks' tensors (framework stream): this response's stream waits for them, which covers what
        # that stream did before
        made = _current_stream() if peers else None
        slot, s, requests = self._begin(group, made, sum(counts) * self.size * dtype_size(first.tensor_dtype))
        if made is not None:
            peers.append(self._wait_for(s, made))
        event = self._acquire(s)
        try:
            plain = first.wire_dtype == first.tensor_dtype
            stays = self.size == 1 and inputs == outputs and plain and first.prescale == first.postscale == 1.0
            if len(group) == 1 and plain and not stays:
                inputs = self._aligned(slot, s, inputs, counts[0], first.tensor_dtype)
            if stays or not any(counts):
                check(lib().hvdhip_event_record(event, s.handle), "hvdhip_event_record")
            elif first.op == ADASUM and self.size > 1:
                self._adasum(slot, s, first, inputs, outputs, counts, event)
            else:
                self._sum(slot, s, first, inputs, outputs, counts, event)
        except Exception:
            self._give_up(s, event)
            raise
        self._finish(s, requests, event, peers)

    def _aligned(self, slot, s, inputs, count, dtype):
        """Foreign memory may lie on addresses that no element type fits.  Alone in its response such a tensor is
        copied as bytes first; fused ones are refused, as they are by a fusion plan."""
        es = dtype_size(dtype)
        if count == 0 or not any(p % es for p in inputs):
            return inputs
        sources, stride = list(dict.fromkeys(inputs)), (count * es + 255) // 256 * 256
        buf = self._buffer(slot, "aligned", len(sources) * stride)
        at = {p: buf + i * stride for i, p in enumerate(sources)}
        as_bytes = TORCH_TO_HVD[torch.uint8]
        H.ranks_sum(list(at.values()), sources, [count * es] * len(sources), 1, as_bytes, as_bytes, as_bytes, 1.0, 1.0, s)
        return [at[p] for p in inputs]

    @staticmethod
    def _acquire(s):
        """An event of the stream's pool for a response's completion."""
        ev = c_void_p()
        check(lib().hvdhip_event_acquire(s.handle, ctypes.byref(ev)), "hvdhip_event_acquire")
        return ev

    @staticmethod
    def _give_up(s, event):
        """For a response that failed after part of it was queued: that part may still read the ranks' tensors and
        write the outputs, which nothing holds on to once the caller has the error."""
        try:
            s.synchronize()
        finally:
            check(lib().hvdhip_event_release(s.handle, event), "hvdhip_event_release")

    def _sum(self, slot, s, req, inputs, outputs, counts, event):
        """outputs = postscale * (sum over ranks of prescale * inputs), in one pass if the outputs lie over no
        other tensor of the response.  The event is bound to the last launch, for callers that wait for handles: a
        small tensor of eight ranks takes 23 us (25 with the event recorded by itself, as an allgather's is); with a
        device-wide synchronization behind each call 35 (29)."""
        tdt, wire = req.tensor_dtype, req.wire_dtype
        if self.size <= H.RANKS_SUM_MAX_WORLD:
            if H.ranks_sum(outputs, inputs, counts, self.size, tdt, wire, tdt, req.prescale, req.postscale, s,
                           event=event):
                return
        offsets, nbytes = self._offsets(counts, wire)
        buf = self._to_buffer(slot, s, req, inputs, counts, offsets, nbytes)
        self._from_buffer(buf, s, req, outputs, counts, offsets, event)

    @staticmethod
    def _offsets(counts, dtype):
        """Byte offset of every entry in a fusion buffer and the buffer's length: each entry padded to 16
        bytes (ops/gpu_operations.cc:141)."""
        es, at, offsets = dtype_size(dtype), 0, []
        for n in counts:
            offsets.append(at)
            at += (n * es + 15) // 16 * 16
        return offsets, at

    def _to_buffer(self, slot, s, req, inputs, counts, offsets, nbytes, which=0):
        """The sum of the ranks' scaled tensors in one of the stream slot's buffers."""
        tdt, wire, n = req.tensor_dtype, req.wire_dtype, len(counts)
        buf = self._buffer(slot, which, nbytes)
        head = min(len(inputs) // n, H.RANKS_SUM_MAX_WORLD)
        H.ranks_sum([buf + o for o in offsets], inputs[:head * n], counts, head, tdt, wire, wire, req.prescale, 1.0, s,
                    pad=True)
        for at in range(head * n, len(inputs), n):  # more ranks than one pass takes: one by one
            one = self._buffer(slot, 1, nbytes)
            H.ranks_sum([one + o for o in offsets], inputs[at:at + n], counts, 1, tdt, wire, wire, req.prescale, 1.0, s,
                        pad=True)
            H.reduce_sum(buf, one, nbytes // dtype_size(wire), wire, s)
        return buf

    def _from_buffer(self, buf, s, req, outputs, counts, offsets, event):
        tdt, wire = req.tensor_dtype, req.wire_dtype
        if H.ranks_sum(outputs, [buf + o for o in offsets], counts, 1, wire, wire, tdt, 1.0, req.postscale, s,
                       event=event):
            return
        for out, o, n in zip(outputs, offsets, counts):  # outputs that share memory: in order
            H.ranks_sum([out], [buf + o], [n], 1, wire, wire, tdt, 1.0, req.postscale, s)
        check(lib().hvdhip_event_record(event, s.handle), "hvdhip_event_record")

    def _wait_for(self, s, producer, event=None):
        """Makes the stream wait for what the framework's stream `producer` holds now, if there is anything, or for
        `event`, which was recorded there.  Returns the event that it waits for."""
        if event is None:
            if self.busy.get(producer, 0) < self.cycles:
                if producer == _current_stream():
                    handle = torch._C._cuda_getCurrentRawStream(producer[1])
                else:
                    handle = _stream_of(producer).cuda_stream
                idle = c_int()
                check(lib().hvdhip_stream_idle(handle, ctypes.byref(idle)), "hvdhip_stream_idle")
                if idle.value:
                    return None
                if len(self.busy) > 64:
                    self.busy.clear()
                self.busy[producer] = self.cycles + _BUSY_CYCLES
            event = torch.cuda.Event()
            event.record(_stream_of(producer))
        check(lib().hvdhip_stream_wait_event(s.handle, c_void_p(event.cuda_event)), "hvdhip_stream_wait_event")
        return event

    def _begin(self, group, made=None, nbytes=0):
        """Picks the stream slot of a fused response and makes it wait for the framework's streams that its requests were
        enqueued on, all but the one that the caller makes it wait for (`made`).  nbytes: what it reads."""
        self.responses += 1
        slot = self.slot
        if nbytes >= _BYTES_OF_ITS_OWN:
            self.staying = self.cycles
        if self.staying != self.cycles:
            self.slot = (slot + 1) % len(self.streams)
        s = self.streams[slot]
        requests, producers = _front.requests(group)
        for producer in producers:
            if producer != made:
                self.ready[producer] = self._wait_for(s, producer, self.ready.get(producer))
        return slot, s, requests

    @staticmethod
    def _finish(s, requests, event, keepalive=None):
        _front.attach(requests, Marker(s, event, len(requests), keepalive))

    def _execute_allgather(self, group):
        """The fusion-buffer side of a fused allgather (AllgatherOp::MemcpyInFusionBuffer /
        MemcpyOutFusionBuffer, ops/collective_operations.cc:234-288): entry e of rank r goes to row
        offset sum(first dimensions of ranks < r) of output e.  Every rank's rows sit in this GPU's
        memory, so they are copied straight there, the buffer in between left out."""
        slot, s, requests = self._begin(group)
        dtype = group[0][0].tensor_dtype
        es = dtype_size(dtype)
        places, sources, counts = _front.places(group, es)
        if any(p % es for p in sources):  # foreign memory that no element type fits: bytes
            counts, dtype = [n * es for n in counts], TORCH_TO_HVD[torch.uint8]
        event = self._acquire(s)
        try:
            if not H.ranks_sum(places, sources, counts, 1, dtype, dtype, dtype, 1.0, 1.0, s):
                raise RuntimeError("an allgather's output lies over one of its inputs")
            # recorded by itself: bound to the copy's launch it saves 2 us here, and costs 6 in a device-wide
            # synchronization that follows, as scripts that read the rows on the host do
            check(lib().hvdhip_event_record(event, s.handle), "hvdhip_event_record")
        except Exception:
            self._give_up(s, event)
            raise
        self._finish(s, requests, event)

    def _adasum(self, slot, s, req, inputs, outputs, counts, event):
        """Ranks of one node are summed (the reduce-scatter leg of
        ops/adasum_gpu_operations.cc:174-197), then the node results are combined pairwise at
        distances 1, 2, 4 ... like the levels of Adasum::FusedAllreduce (ops/adasum/adasum.h:194-340)."""
        tdt, wire, L, nodes = req.tensor_dtype, req.wire_dtype, self.local_size, self.size // self.local_size
        if nodes == 1:
            return self._sum(slot, s, req, inputs, outputs, counts, event)
        offsets, nbytes = self._offsets(counts, wire)
        source, prescale = tdt, req.prescale
        if L > 1:
            ranks = L * len(counts)
            sums = [self._to_buffer(slot, s, req, inputs[node * ranks:(node + 1) * ranks], counts, offsets, nbytes,
                                    2 + node) for node in range(nodes)]
            inputs, source, prescale = [b + o for b in sums for o in offsets], wire, 1.0
        space = H.adasum_ranks_workspace(counts, nodes, wire)
        work = self._buffer(slot, "adasum", space)
        # Two nodes are two launches, and the event is recorded by itself as in an allgather: 4 million fp32 37 us either
        # way, and with a device-wide synchronization behind the call 41 (48 with the event bound to the last launch).
        # Eight nodes take 109 and 121 with the event bound, 112 and 138 without.
        bound = event if nodes > 2 else None
        if H.adasum_ranks(outputs, inputs, counts, nodes, source, wire, tdt, prescale, req.postscale, work, space, s,
                          event=bound):
            if bound is None:
                check(lib().hvdhip_event_record(event, s.handle), "hvdhip_event_record")
            return
        buf = self._buffer(slot, 0, nbytes)  # outputs that share memory with other tensors
        H.adasum_ranks([buf + o for o in offsets], inputs, counts, nodes, source, wire, wire, prescale, 1.0, work, space, s)
        self._from_buffer(buf, s, req, outputs, counts, offsets, event)

    # ---- completion -----------------------------------------------------

    @staticmethod
    def _release(marker):
        check(lib().hvdhip_event_release(marker.stream.handle, marker.event), "hvdhip_event_release")

    def poll(self, request):
        if not request.submitted:
            if not self.cycling.acquire(blocking=False):
                return False  # in another thread's cycle, or in the next
            try:
                self.run_cycle()
            finally:
                self.cycling.release()
            if not request.submitted:
                return False  # asked from within its own cycle
        if request.error is not None:
            return True
        for m in request.markers:
            done = c_int()
            check(lib().hvdhip_event_query(m.event, ctypes.byref(done)), "hvdhip_event_query")
            if not done.value:
                return False
        return True

    def wait(self, request):
        if not request.submitted:
            self.run_cycle()
            if not request.submitted:  # still in flight, and the tensor as it was
                raise HorovodInternalError("An operation cannot be waited for from within its own cycle before its response.")
        try:
            for m in request.markers:
                if not m.done:
                    check(lib().hvdhip_event_synchronize(m.event), "hvdhip_event_synchronize")
                    m.done, m.keepalive = True, None
        finally:
            for m in request.markers:
                m.refs -= 1
                if m.refs == 0:  # the last request of the response hands the event back to its pool
                    self._release(m)
            request.markers = []
            for e in request.entries:
                self.inflight.pop(e.name, None)
        if request.error is not None:
            raise HorovodInternalError(str(request.error)) from request.error

    def shutdown(self):
        for r in set(self.inflight.values()):
            try:
                self.wait(r)
            except HorovodInternalError:
                pass
        for s in self.streams:
            s.destroy()
        self.streams, self.buffers = [], {}
