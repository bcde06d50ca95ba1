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
from ctypes import c_int, c_int64, c_void_p

import torch

from .. import host as H
from .._lib import adapter_lib, check, dtype_size, lib

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


class HorovodInternalError(RuntimeError):
    """An error of the op layer surfacing in the caller (horovod/common/exceptions.py:18-23)."""


class Entry:
    __slots__ = ("name", "tensor", "output", "count", "parts")

    def __init__(self, name, tensor, output):
        self.name, self.tensor, self.output, self.count = name, tensor, output, tensor.numel()
        self.parts = None  # allgather: what every rank contributes, rank 0 first


class Request:
    __slots__ = ("kind", "entries", "op", "prescale", "postscale", "divisor", "tensor_dtype", "wire_dtype", "device",
                 "producer", "markers", "submitted", "error", "grouped")

    def __init__(self, entries, op, prescale, postscale, divisor, tensor_dtype, wire_dtype, device,
                 kind="allreduce", grouped=False):
        self.kind = kind
        self.entries = entries
        self.op, self.prescale, self.postscale, self.divisor = op, float(prescale), float(postscale), divisor
        self.tensor_dtype, self.wire_dtype, self.device = tensor_dtype, wire_dtype, device
        self.producer = None     # the framework stream that was current at enqueue (torch's identifiers)
        self.markers = []        # one Marker per fused response that carries one of the entries
        self.submitted = False
        self.error = None
        self.grouped = grouped

    def key(self):
        return (self.kind, self.op, self.device, self.tensor_dtype, self.wire_dtype, self.prescale, self.postscale)


class Marker:
    """Completion event of one fused response, shared by the requests it carried
    (ops/gpu_operations.cc:50-56 records one per response)."""
    __slots__ = ("stream", "event", "refs", "done", "keepalive")

    def __init__(self, stream, event, refs, keepalive):
        self.stream, self.event, self.refs = stream, event, refs
        self.done = False
        self.keepalive = keepalive  # the other ranks' tensors, until the response has completed


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
        self.queue = []
        self.inflight = {}       # tensor name -> request, until synchronised
        self.buffers = {}        # (slot, what for) -> torch uint8 tensor
        self.cycles = 0
        self.responses = 0       # fused responses executed so far
        self.ready = {}          # framework stream -> event recorded during the current cycle

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
            parts = [e.tensor]
            for rank in range(1, self.size):
                t = e.tensor if self.peer_source is None else self.peer_source(rank, e.name, e.tensor)
                if (not isinstance(t, torch.Tensor) or not t.is_cuda or t.dtype != e.tensor.dtype
                        or t.dim() != e.tensor.dim() or t.shape[1:] != e.tensor.shape[1:] or not t.is_contiguous()):
                    self.inflight.pop(e.name, None)
                    raise HorovodInternalError(
                        "Mismatched allgather tensor shapes: ranks may differ in the first dimension only "
                        "(tensor %r)." % e.name)
                parts.append(t)
            e.parts = parts
            e.output.resize_((sum(t.shape[0] for t in parts),) + tuple(e.tensor.shape[1:]))

    def run_cycle(self):
        """Fuses and queues everything enqueued so far (one pass of RunLoopOnce,
        common/operations.cc:593-717, with every request already agreed upon)."""
        pending, self.queue = self.queue, []
        if not pending:
            return
        self.cycles += 1
        self.ready = {}
        flat, sizes, keys, classes = [], [], [], {}
        for r in pending:
            key = classes.setdefault(r.key(), len(classes))
            gathers = r.kind == "allgather"
            es = dtype_size(r.tensor_dtype if gathers else r.wire_dtype)
            for e in r.entries:
                nbytes = (e.output.numel() if gathers else e.count) * es
                if self.batch_d2d_memcopies and not gathers:  # no padding on that path
                    nbytes = (nbytes + 15) // 16 * 16
                flat.append((r, e))
                sizes.append(nbytes)
                keys.append(key)
        n = len(flat)
        group_of = (c_int * n)()
        ngroups = adapter_lib().hvd_adapter_fuse_keyed((c_int64 * n)(*sizes), (c_int * n)(*keys), n,
                                                       self.fusion_threshold, 0, group_of)
        groups = [[] for _ in range(ngroups)]
        for i in range(n):
            groups[group_of[i]].append(flat[i])
        for g in groups:
            try:
                if g[0][0].kind == "allgather":
                    self._execute_allgather(g)
                else:
                    self._execute(g)
            except Exception as exc:  # surfaces in synchronize(), like a Status passed to the callback
                for r, _ in g:
                    r.error = exc
        for r in pending:
            r.submitted = True

    # ---- resources ------------------------------------------------------

    def _buffer(self, slot, what, nbytes):
        t = self.buffers.get((slot, what))
        if t is None or t.numel() < nbytes:
            if t is not None:
                self.streams[slot].synchronize()  # queued kernels may still use the smaller buffer
            t = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")
            self.buffers[(slot, what)] = t
        return t.data_ptr()

    def _peers(self, group, addresses):
        """The tensors that the other ranks pass for a group's entries; their addresses are appended rank by rank."""
        source, dtype, peers = self.peer_source, group[0][1].tensor.dtype, []
        for rank in range(1, self.size):
            for _, e in group:
                t = source(rank, e.name, e.tensor)
                if (not isinstance(t, torch.Tensor) or not t.is_cuda or t.dtype != dtype or t.numel() != e.count
                        or not t.is_contiguous()):
                    raise ValueError("peer_source must return a contiguous device tensor of the shape and dtype of %r"
                                     % e.name)
                peers.append(t)
                addresses.append(t.data_ptr())
        return peers

    # ---- one fused response --------------------------------------------

    def _execute(self, group):
        first = group[0][0]
        counts = [e.count for _, e in group]
        inputs = [e.tensor.data_ptr() for _, e in group]  # rank-major: inputs[rank * len(group) + entry]
        peers = made = None
        if self.peer_source is None:
            inputs *= self.size
        elif self.size > 1:
            # the other ranks' tensors (framework stream); this response's stream waits for them, which
            # covers what that stream did before
            peers = self._peers(group, inputs)
            made = _current_stream()
            peers.append(self._record(made))
        slot, s, requests = self._begin(group, made)
        if made is not None:
            self._wait_for(s, peers[-1])
        outputs = [e.output.data_ptr() for _, e in group]
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
        small tensor of eight ranks takes 45 us (48 with the event recorded by itself, as an allgather's is); with a
        device-wide synchronization behind each call 60 (53)."""
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

    @staticmethod
    def _record(producer):
        ev = torch.cuda.Event()
        stream_id, device_index, device_type = producer
        ev.record(torch.cuda.Stream(stream_id=stream_id, device_index=device_index, device_type=device_type))
        return ev

    @staticmethod
    def _wait_for(s, ev):
        check(lib().hvdhip_stream_wait_event(s.handle, c_void_p(ev.cuda_event)), "hvdhip_stream_wait_event")

    def _begin(self, group, covered=None):
        """Picks the stream slot of a fused response and makes it wait for the framework's streams, all but
        the one that the caller makes it wait for."""
        self.responses += 1
        slot, self.slot = self.slot, (self.slot + 1) % len(self.streams)
        s = self.streams[slot]
        requests = list(dict.fromkeys(r for r, _ in group))
        for producer in {r.producer for r in requests}:
            if producer == covered:
                continue
            if producer not in self.ready:
                self.ready[producer] = self._record(producer)
            self._wait_for(s, self.ready[producer])
        return slot, s, requests

    @staticmethod
    def _finish(s, requests, event, keepalive=None):
        marker = Marker(s, event, len(requests), keepalive)
        for r in requests:
            r.markers.append(marker)

    def _execute_allgather(self, group):
        """The fusion-buffer side of a fused allgather (AllgatherOp::MemcpyInFusionBuffer /
        MemcpyOutFusionBuffer, ops/collective_operations.cc:234-288): entry e of rank r goes to row
        offset sum(first dimensions of ranks < r) of output e.  Every rank's rows sit in this GPU's
        memory, so they are copied straight there, the buffer in between left out."""
        slot, s, requests = self._begin(group)
        dtype = group[0][0].tensor_dtype
        es = dtype_size(dtype)
        sources, places, counts = [], [], []
        for _, e in group:
            at = e.output.data_ptr()
            for part in e.parts:
                n = part.numel()
                if n:
                    sources.append(part.data_ptr())
                    places.append(at)
                    counts.append(n)
                    at += n * es
        if any(p % es for p in sources):  # foreign memory that no element type fits: bytes
            counts, dtype = [n * es for n in counts], TORCH_TO_HVD[torch.uint8]
        event = self._acquire(s)
        try:
            if not H.ranks_sum(places, sources, counts, 1, dtype, dtype, dtype, 1.0, 1.0, s):
                raise RuntimeError("an allgather's output lies over one of its inputs")
            # recorded by itself: bound to the copy's launch it saves 3 us here, and costs 17 in a device-wide
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
        # Two nodes are two launches, and the event is recorded by itself as in an allgather: 4 million fp32 66 us either
        # way, and with a device-wide synchronization behind the call 70 (79 with the event bound to the last launch).
        # Eight nodes take 101 and 115 with the event bound, 106 and 128 without.
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

    def poll(self, request):
        if not request.submitted:
            self.run_cycle()
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
        try:
            for m in request.markers:
                if not m.done:
                    check(lib().hvdhip_event_synchronize(m.event), "hvdhip_event_synchronize")
                    m.done, m.keepalive = True, None
        finally:
            for m in request.markers:
                m.refs -= 1
                if m.refs == 0:  # the last request of the response hands the event back to its pool
                    check(lib().hvdhip_event_release(m.stream.handle, m.event), "hvdhip_event_release")
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
