"""What the gradient path is timed on: a dozen calls as users of the framework make them, and draw() for
more of the same ranges.

Two kinds of users are covered.  A training script sees ``horovod_amd.torch``: it averages a metric, hands
over every gradient of a backward pass (by itself, through the optimizer or as a group, with and without
fp16 compression), an Adasum delta, the rows of a sparse gradient.  It runs as rank 0 of a world of eight whose other ranks hold values of their
own.  An op layer written in C++ sees the C ABI: pack a fused response, sum the incoming chunks, unpack,
combine two vectors by Adasum, scale or copy what is not fused.  It owns the fusion buffers (one per stream
slot, for the life of the job) and the plans.  Sizes are those of the repository's own workloads (ResNet-50,
BERT-large, GPT-2 XL gradients, the small-tensor stress set, the Adasum vectors) and of generic mixes.
"""
import math
import random

import torch

import horovod_amd.torch as hvd
from horovod_amd import DTYPE, AdasumPlan, FusionPlan, Stream
from horovod_amd import host as H
from horovod_amd import workloads as W

WORLD = 8
TORCH = {"uint8": torch.uint8, "int8": torch.int8, "int32": torch.int32, "int64": torch.int64,
         "float16": torch.float16, "float32": torch.float32, "float64": torch.float64}
SIZE = {"uint8": 1, "int8": 1, "int32": 4, "int64": 8, "float16": 2, "float32": 4, "float64": 8}


def listed():
    return [
        # loss and accuracy averaged over the ranks at the end of a step: nothing but latency
        {"name": "metric_average", "kind": "metric", "n": 2, "dtype": "float32"},
        # the 161 gradients of ResNet-50, handed over one by one as the optimizer's hooks do, in place
        {"name": "resnet50_gradients", "kind": "gradients", "set": "resnet50", "dtype": "float32"},
        # BERT-large under DistributedOptimizer with fp16 compression, up to the averaged gradients (where
        # a script clips them before the update): the largest step
        {"name": "bert_large_optimizer_fp16", "kind": "optimizer", "set": "bert_large", "dtype": "float32", "fp16": True},
        # one BERT-large encoder layer's update combined by Adasum over eight nodes
        {"name": "adasum_delta", "kind": "adasum_delta", "set": "bert_layer", "dtype": "float32"},
        # a sparse embedding gradient: the touched rows and their indices, a different number on every rank
        {"name": "sparse_rows", "kind": "rows", "rows": 2041, "width": 1024, "dtype": "float32"},
        # op layer: ResNet-50's two fusion cycles on one stream, summed with one other buffer
        {"name": "cycles_resnet50", "kind": "cycles", "set": "resnet50", "dtype": "float32", "wire": "float32",
         "peers": 1, "streams": 1, "arrays": False},
        # op layer: 1,024 small tensors into the fusion buffer and out again
        {"name": "cycles_small_tensors", "kind": "cycles", "set": "stress", "dtype": "float32", "wire": "float32",
         "peers": 0, "streams": 1, "arrays": False},
        # op layer: four layers of GPT-2 XL in fp16 over two streams, through the calls that take arrays
        {"name": "copies_gpt2_fp16", "kind": "cycles", "set": "gpt2_layers", "dtype": "float16", "wire": "float16",
         "peers": 1, "streams": 2, "arrays": True},
        # one GPU's eighth of a 62 MiB fp16 buffer, seven incoming chunks
        {"name": "share_sum_fp16", "kind": "share", "n": 4067712, "peers": 7, "dtype": "float16"},
        # Adasum of two vectors of 2^25 elements in 64 layers of very different lengths
        {"name": "adasum_64_layers", "kind": "combine", "n": 1 << 25, "layers": 64, "mix": 13, "dtype": "float32"},
        # Adasum of a small network: many layers, most of them a few hundred elements
        {"name": "adasum_small_layers", "kind": "combine", "n": 270011, "layers": 61, "mix": 5, "dtype": "float16"},
        # a tensor larger than the fusion threshold (GPT-2 XL's embedding): scaled by itself, not packed
        {"name": "scale_embedding_fp16", "kind": "scale", "n": 50257 * 1600, "dtype": "float16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["metric", "gradients", "optimizer", "grouped", "adasum_delta", "rows", "cycles", "share",
                       "combine", "scale"])
    mix = rng.randrange(1 << 30)
    if kind == "metric":
        return {"kind": kind, "n": _log(rng, 1, 4096), "dtype": rng.choice(["float32", "float64"])}
    if kind in ("gradients", "optimizer", "grouped", "adasum_delta", "cycles"):
        tensors = _log(rng, 1, 60 if kind == "grouped" else 320)
        total = _log(rng, tensors * 200, 40 << 20)
        case = {"kind": kind, "set": "mix", "tensors": tensors, "total": total, "mix": mix, "dtype": "float32"}
        if kind == "gradients":
            case["dtype"] = rng.choice(["float32", "float16"])
        elif kind in ("optimizer", "grouped"):
            case["fp16"] = rng.choice([True, False])
        elif kind == "adasum_delta":
            case["dtype"] = rng.choice(["float32", "float16", "float64"])
        elif kind == "cycles":
            case["dtype"] = rng.choice(["float32", "float16", "float64"])
            case["wire"] = rng.choice(["float16", "float32"]) if case["dtype"] == "float32" else case["dtype"]
            case["peers"] = rng.choice([0, 1, 3, 7])
            case["streams"] = rng.choice([1, 2])
            case["arrays"] = case["wire"] == case["dtype"] and rng.random() < 0.3
        return case
    if kind == "rows":
        width = rng.choice([1, 64, 300, 1024, 1600])
        return {"kind": kind, "rows": max(1, _log(rng, 64, 8 << 20) // width), "width": width,
                "dtype": rng.choice(["float32", "float16", "int64"])}
    if kind == "share":
        return {"kind": kind, "n": _log(rng, 1000, 32 << 20), "peers": rng.choice([1, 2, 3, 7, 7, 15]),
                "dtype": rng.choice(["float16", "float32", "float64", "int32", "uint8"])}
    if kind == "combine":
        layers = _log(rng, 1, 400)
        return {"kind": kind, "n": _log(rng, layers * 100, 40 << 20), "layers": layers, "mix": mix,
                "dtype": rng.choice(["float16", "float32", "float64"])}
    return {"kind": kind, "n": _log(rng, 1000, 96 << 20),
            "dtype": rng.choice(["float16", "float32", "float64", "int32", "int64", "uint8", "int8"])}


# ---- sizes ---------------------------------------------------------------------------------------

def _parts(total, n, mix):
    """total cut into n parts of very different size (each at least 1), odd ones among them."""
    rng = random.Random(mix)
    weights = [math.exp(rng.uniform(0.0, math.log(3000.0))) for _ in range(n)]
    scale = (total - n) / sum(weights)
    parts = [1 + int(w * scale) for w in weights]
    parts[parts.index(max(parts))] += total - sum(parts)
    return parts


def _counts(case):
    """Element counts of the tensors of a case."""
    what = case["set"]
    if what == "mix":
        return _parts(case["total"], case["tensors"], case["mix"])
    if what == "stress":
        return W.stress_counts()
    shapes = {"resnet50": W.resnet50_shapes, "bert_large": W.bert_large_shapes,
              "bert_layer": lambda: W.bert_large_shapes()[5:21],
              "gpt2_layers": lambda: W.gpt2_xl_shapes()[2:50]}[what]()
    return [W.numel(s) for s in shapes]


def _layers(case):
    return W.adasum_layer_counts(case["n"], case["layers"], case["mix"])


def _rank_rows(case):
    """Rows that each rank contributes: up to a tenth apart."""
    return [max(1, case["rows"] + (r * 37) % 23 * case["rows"] // 200) for r in range(WORLD)]


# ---- what a program holds ------------------------------------------------------------------------

_kept = {}   # streams and fusion buffers: one per slot for the life of the job, whatever runs there
_peers = {}  # operation name -> what ranks 1..WORLD-1 pass under it


def _peer_source(rank, name, tensor):
    return _peers[name][rank - 1]


def _hvd():
    if not hvd.is_initialized():
        hvd.init(size=WORLD, peer_source=_peer_source)


def _stream(slot):
    if ("stream", 0) not in _kept:
        for i in range(2):
            _kept["stream", i] = Stream()
    return _kept["stream", slot]


def _fusion_buffer(slot, nbytes):
    t = _kept.get(("buffer", slot))
    if t is None or t.numel() < nbytes:
        torch.cuda.synchronize()
        t = _kept["buffer", slot] = torch.zeros(max(nbytes, W.FUSION_THRESHOLD), dtype=torch.uint8, device="cuda")
    return t.data_ptr()


class State:
    """Inputs, outputs and handles of one case; plans go back to the library and peers are forgotten with it."""
    count = 0

    def __init__(self, case):
        self.case = case
        self.plans, self.names = [], []
        State.count += 1
        self.id = State.count

    def peers_of(self, name, tensors):
        _peers[name] = tensors
        self.names.append(name)

    def __del__(self):
        try:
            for p in self.plans:
                p.destroy()
            for n in self.names:
                _peers.pop(n, None)
        except Exception:  # the interpreter is going down
            pass


def _views(counts, dtype):
    """Tensors of the given counts inside one allocation, each on a 512-byte boundary as the framework's
    allocator places them: (the whole, its tensors)."""
    step = 512 // SIZE[dtype]
    at, offs = 0, []
    for c in counts:
        offs.append(at)
        at += (c + step - 1) // step * step
    whole = torch.zeros(max(at, 1), dtype=TORCH[dtype], device="cuda")
    return whole, [whole[o:o + c] for o, c in zip(offs, counts)]


def _fill(t, gen):
    """Gradient-like values: zero mean, about 0.01; integers over a small range."""
    if t.is_floating_point():
        return t.normal_(0.0, 0.01, generator=gen)
    return t.random_(0, 100, generator=gen)


def _inputs(counts, dtype, gen):
    whole, views = _views(counts, dtype)
    _fill(whole, gen)
    return whole, views


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    s = State(case)
    kind, dtype = case["kind"], case["dtype"]
    code = DTYPE[dtype]
    if kind == "metric":
        _hvd()
        s.value = _fill(torch.empty(case["n"], dtype=TORCH[dtype], device="cuda"), gen)
        s.name = "metric.%d" % s.id
        s.peers_of("allreduce." + s.name, [_fill(torch.empty_like(s.value), gen) for _ in range(WORLD - 1)])
    elif kind in ("gradients", "optimizer", "grouped", "adasum_delta"):
        _hvd()
        counts = _counts(case)
        s.whole, s.tensors = _inputs(counts, dtype, gen)
        peers = [_inputs(counts, dtype, gen)[1] for _ in range(WORLD - 1)]
        s.compression = hvd.Compression.fp16 if case.get("fp16") else hvd.Compression.none
        if kind == "grouped":
            s.name = "group.%d" % s.id
            names = ["grouped_allreduce.%s_%dof%d" % (s.name, i + 1, len(counts)) for i in range(len(counts))]
        else:
            s.ops = ["grad.%d.%d" % (s.id, i) for i in range(len(counts))]
            names = ["allreduce." + n for n in s.ops]
        for i, name in enumerate(names):
            s.peers_of(name, [p[i] for p in peers])
        if kind == "optimizer":
            params = [torch.nn.Parameter(v) for v in _views(counts, dtype)[1]]
            for p, g in zip(params, s.tensors):
                p.grad = g
            s.opt = hvd.DistributedOptimizer(torch.optim.SGD(params, lr=0.01), named_parameters=zip(s.ops, params),
                                             compression=s.compression)
    elif kind == "rows":
        _hvd()
        rows = _rank_rows(case)
        s.values = [_fill(torch.empty(r, case["width"], dtype=TORCH[dtype], device="cuda"), gen) for r in rows]
        s.indices = [torch.randint(0, 1 << 20, (r, 1), generator=gen, device="cuda") for r in rows]
        s.ops = ["values.%d" % s.id, "indices.%d" % s.id]
        s.peers_of("allgather." + s.ops[0], s.values[1:])
        s.peers_of("allgather." + s.ops[1], s.indices[1:])
    elif kind == "cycles":
        counts, wire = _counts(case), case["wire"]
        s.whole, tensors = _inputs(counts, dtype, gen)
        s.out, outs = _views(counts, dtype)
        s.cycles = []
        for g in W.fuse([c * SIZE[wire] for c in counts]):
            plan = FusionPlan([tensors[i].data_ptr() for i in g], [outs[i].data_ptr() for i in g],
                              [counts[i] for i in g], code, DTYPE[wire])
            s.plans.append(plan)
            n = plan.buffer_len // SIZE[wire]
            peers = [_fill(torch.empty(n, dtype=TORCH[wire], device="cuda"), gen) for _ in range(case["peers"])]
            arrays = None
            if case["arrays"]:
                arrays = ([tensors[i].data_ptr() for i in g], [outs[i].data_ptr() for i in g],
                          [counts[i] * SIZE[dtype] for i in g], plan.offsets())
            s.cycles.append((plan, n, peers, arrays))
        s.slots = [(_stream(i), _fusion_buffer(i, max(p.buffer_len for p in s.plans))) for i in range(case["streams"])]
    elif kind == "share":
        n = case["n"]
        s.resident = _fill(torch.empty(n, dtype=TORCH[dtype], device="cuda"), gen)
        s.staging = [_fill(torch.empty(n, dtype=TORCH[dtype], device="cuda"), gen) for _ in range(case["peers"])]
    elif kind == "combine":
        s.a = _fill(torch.empty(case["n"], dtype=TORCH[dtype], device="cuda"), gen)
        s.b = _fill(torch.empty(case["n"], dtype=TORCH[dtype], device="cuda"), gen).add_(s.a, alpha=0.3)
        s.plan = AdasumPlan(_layers(case), code)
        s.plans.append(s.plan)
    else:
        s.src = _fill(torch.empty(case["n"], dtype=TORCH[dtype], device="cuda"), gen)
        s.dst = torch.zeros_like(s.src)
    return s


def _run_cycles(s):
    case = s.case
    code, wire = DTYPE[case["dtype"]], DTYPE[case["wire"]]
    for i, (plan, n, peers, arrays) in enumerate(s.cycles):
        stream, buf = s.slots[i % len(s.slots)]
        if arrays:
            tensors, outs, sizes, offsets = arrays
            at = [buf + o for o in offsets]
            H.batched_scaled_d2d_memcpy(at, tensors, sizes, 1.0 / WORLD, code, stream)
        else:
            plan.pack(buf, 1.0 / WORLD, stream)
        if peers:
            H.reduce_sum_k(buf, [p.data_ptr() for p in peers], n, wire, stream)
        if arrays:
            H.batched_scaled_d2d_memcpy(outs, at, sizes, 0.5, code, stream)
        else:
            plan.unpack(buf, 0.5, stream)
    return s.out


def run(state):
    s, kind = state, state.case["kind"]
    if kind == "metric":
        return hvd.allreduce(s.value, name=s.name)
    if kind in ("gradients", "adasum_delta"):
        op = hvd.Adasum if kind == "adasum_delta" else hvd.Average
        handles = [hvd.allreduce_async_(t, name=n, op=op) for t, n in zip(s.tensors, s.ops)]
        for h in handles:
            hvd.synchronize(h)
        return s.whole
    if kind == "optimizer":
        s.opt.synchronize()
        return s.whole
    if kind == "grouped":
        return hvd.grouped_allreduce(s.tensors, name=s.name, compression=s.compression)
    if kind == "rows":
        handles = [hvd.allgather_async(s.values[0], name=s.ops[0]), hvd.allgather_async(s.indices[0], name=s.ops[1])]
        return [hvd.synchronize(h) for h in handles]
    if kind == "cycles":
        return _run_cycles(s)
    if kind == "share":
        H.reduce_sum_k(s.resident.data_ptr(), [p.data_ptr() for p in s.staging], s.case["n"], DTYPE[s.case["dtype"]],
                       _stream(0))
        return s.resident
    if kind == "combine":
        s.plan.combine(s.a.data_ptr(), s.b.data_ptr(), _stream(0))
        return s.a
    H.scale_buffer(s.src.data_ptr(), s.dst.data_ptr(), s.case["n"], 1.0 / WORLD, DTYPE[s.case["dtype"]], _stream(0))
    return s.dst


# ---- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    flops = 0
    if kind in ("metric", "gradients", "optimizer", "grouped", "adasum_delta"):
        # every rank's tensors in, this rank's result out
        n = case["n"] if kind == "metric" else sum(_counts(case))
        nbytes = (WORLD + 1) * n * es
        flops = WORLD * n if kind != "adasum_delta" else (WORLD - 1) * 9 * n
    elif kind == "rows":
        n = sum(_rank_rows(case))
        nbytes = 2 * n * (case["width"] * es + 8)
    elif kind == "cycles":
        # The calls of a cycle are separate, with the collective between them in a real job: the fusion
        # buffer is each call's output and the next one's input.
        n, ws, k = sum(_counts(case)), SIZE[case["wire"]], case["peers"]
        nbytes = 2 * n * (es + ws) + ((k + 2) * n * ws if k else 0)
        flops = (2 + k) * n
    elif kind == "share":
        nbytes = (case["peers"] + 2) * case["n"] * es
        flops = case["peers"] * case["n"]
    elif kind == "combine":
        # both vectors in, one out; the coefficients need all of a layer before any of it is written
        nbytes = 3 * case["n"] * es
        flops = 9 * case["n"]
    else:
        nbytes = 2 * case["n"] * es
        flops = case["n"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Copies, scales and sums are defined to the bit: one rounding per scale and one after every rank's
    summand, in rank order.  Adasum's sums are taken in double in an order that is left open.  Taken in another
    order (4 KiB in place of 16 KiB per partial sum, three passes) the float64 results moved by 2e-16 (norm) and
    1e-15 (largest), and no float32 or float16 element of 34 million moved; there the bound is a unit in the last
    place of a few elements, as where a coefficient's last bit tips a rounding."""
    if case["kind"] not in ("combine", "adasum_delta"):
        return "exact"
    return {"float16": {"rel": 2e-5, "max": 2e-3}, "float32": {"rel": 1e-8, "max": 3e-7},
            "float64": {"rel": 1e-15, "max": 4e-15}}[case["dtype"]]
