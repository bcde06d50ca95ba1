"""hvdhip_ranks_sum against the oracle's scale -> sum -> scale at the edges of its chunks (4 KiB), rows per
launch (64, or fewer for many ranks) and ranks per batch (8)."""
import numpy as np
import pytest
import torch

from horovod_amd import DTYPE
from horovod_amd import host as H

pytestmark = pytest.mark.gpu

NP = {"uint8": np.uint8, "int8": np.int8, "int16": np.int16, "int32": np.int32, "int64": np.int64,
      "float16": np.float16, "float32": np.float32, "float64": np.float64}


def _values(rng, n, dtype):
    if dtype.startswith("float"):
        return rng.uniform(-2, 2, n).astype(NP[dtype])
    return rng.integers(0, 120, n).astype(NP[dtype])


def _expected(orc, ranks, dtype, wire, pre, post):
    code = DTYPE[wire]
    acc = None
    for v in ranks:
        w = v.astype(np.float16) if wire != dtype else v
        w = orc.scale_buffer(w, pre, code) if pre != 1.0 else w
        acc = w if acc is None else orc.sum(w, acc.copy(), code)
    acc = orc.scale_buffer(acc, post, code) if post != 1.0 else acc
    return acc.astype(NP[dtype])


@pytest.mark.parametrize("dtype,wire", [(d, d) for d in NP] + [("float32", "float16")])
@pytest.mark.parametrize("world", [1, 2, 7, 8, 9, 20])
def test_ranks_sum_equals_scale_sum_scale(gpu, orc, dtype, wire, world):
    rng = np.random.default_rng(world)
    tile = 4096 // np.dtype(NP[dtype]).itemsize
    counts = [1, 0, 3, tile - 1, tile, tile + 1, 5 * tile + 7, 255] + [int(x) for x in rng.integers(1, 40, 70)]
    pre, post = (1.0, 1.0) if dtype == "int16" else ((0.125, 0.3) if world % 2 else (1.0, 0.7))
    host = [[_values(rng, c, dtype) for c in counts] for _ in range(world)]
    # one element into the allocation each: only element alignment is promised
    dev = [[torch.from_numpy(np.concatenate([v[:1], v])).cuda()[1 if v.size else 0:] for v in rank] for rank in host]
    out = [torch.zeros(c + 1, dtype=dev[0][0].dtype, device="cuda") for c in counts]
    torch.cuda.synchronize()
    code, wcode = DTYPE[dtype], DTYPE[wire]
    assert H.ranks_sum([o.data_ptr() for o in out], [t.data_ptr() for r in dev for t in r], counts, world, code, wcode,
                       code, pre, post, gpu.stream)
    # in place as well: rank 0's tensors are the outputs
    mine = [t.data_ptr() for t in dev[0]]
    assert H.ranks_sum(mine, [t.data_ptr() for r in dev for t in r], counts, world, code, wcode, code, pre, post,
                       gpu.stream)
    gpu.stream.synchronize()
    for i, c in enumerate(counts):
        if c == 0:
            continue
        want = _expected(orc, [host[r][i] for r in range(world)], dtype, wire, pre, post)
        got = out[i].cpu().numpy()
        assert np.array_equal(got[:c].view(np.uint8), want.view(np.uint8)), (i, c)
        assert got[c] == 0, "wrote behind its tensor"
        assert np.array_equal(dev[0][i].cpu().numpy().view(np.uint8), want.view(np.uint8)), (i, c)


@pytest.mark.parametrize("dtype,wire", [(d, d) for d in ("uint8", "float16", "float32", "float64")] + [("float32", "float16")])
@pytest.mark.parametrize("world", [3, 4, 5, 6, 7, 8])
def test_ranks_sum_at_the_edges_of_split_tiles(gpu, orc, dtype, wire, world):
    """Tiles of 64 and 128 vectors, the ranks over two or four wavefronts of which the last may have one rank."""
    rng = np.random.default_rng(10 + world)
    vec = 16 // np.dtype(NP[dtype]).itemsize
    counts = [vec - 1, vec, 63 * vec + 1] + [t * vec + d for t in (64, 128, 192, 256) for d in (-1, 0, 1)] + [9999]
    counts = [max(1, c) for c in counts]
    host = [[_values(rng, c, dtype) for c in counts] for _ in range(world)]
    dev = [[torch.from_numpy(np.concatenate([v[:1], v])).cuda()[1:] for v in rank] for rank in host]
    code, wcode = DTYPE[dtype], DTYPE[wire]
    offs = np.cumsum([0] + [(c * np.dtype(NP[dtype]).itemsize + 15) // 16 * 16 for c in counts])
    buf = torch.full((int(offs[-1]) + 16,), 255, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    assert H.ranks_sum([buf.data_ptr() + int(o) for o in offs[:-1]], [t.data_ptr() for r in dev for t in r], counts, world,
                       code, wcode, code, 0.5, 0.3, gpu.stream, pad=True)
    gpu.stream.synchronize()
    image = buf.cpu().numpy()
    assert (image[offs[-1]:] == 255).all(), "wrote behind the buffer"
    for i, c in enumerate(counts):
        want = _expected(orc, [host[r][i] for r in range(world)], dtype, wire, 0.5, 0.3).view(np.uint8)
        piece = image[offs[i]:offs[i + 1]]
        assert np.array_equal(piece[:want.size], want) and not piece[want.size:].any(), (i, c)


@pytest.mark.parametrize("dtype,wire", [("uint8", "uint8"), ("int64", "int64"), ("float16", "float16"), ("float32", "float32"),
                                        ("float64", "float64"), ("float32", "float16")])
@pytest.mark.parametrize("world", [9, 10, 11, 12, 15, 16, 17, 23, 31, 64, 255, 256])
def test_ranks_sum_in_batches_of_eight_four_two_and_one(gpu, orc, dtype, wire, world):
    """Every remainder of the ranks beyond eight, for whole vectors and for the elements behind the last; factors that
    are no powers of two, so that a product that was not rounded before its addition would show."""
    rng = np.random.default_rng(world)
    vec = 16 // np.dtype(NP[dtype]).itemsize
    counts = [1, vec, vec + 1, 2 * vec - 1, 256 * vec + vec - 1, 300]
    pre, post = (0.3, 0.7) if dtype.startswith("float") else (1.0, 1.0)
    host = [[_values(rng, c, dtype) for c in counts] for _ in range(world)]
    dev = [[torch.from_numpy(np.concatenate([v[:1], v])).cuda()[1:] for v in rank] for rank in host]
    out = [torch.zeros(c + 1, dtype=dev[0][0].dtype, device="cuda") for c in counts]
    torch.cuda.synchronize()
    code, wcode = DTYPE[dtype], DTYPE[wire]
    assert H.ranks_sum([o.data_ptr() for o in out], [t.data_ptr() for r in dev for t in r], counts, world, code, wcode,
                       code, pre, post, gpu.stream)
    gpu.stream.synchronize()
    for i, c in enumerate(counts):
        want = _expected(orc, [host[r][i] for r in range(world)], dtype, wire, pre, post)
        got = out[i].cpu().numpy()
        assert np.array_equal(got[:c].view(np.uint8), want.view(np.uint8)), (i, c)
        assert got[c] == 0, "wrote behind its tensor"


@pytest.mark.parametrize("dtype", ["uint8", "int8", "int16", "int32", "int64"])
@pytest.mark.parametrize("world", [2, 5, 8, 11])
def test_integer_sums_wrap(gpu, dtype, world):
    rng = np.random.default_rng(world)
    info, n = np.iinfo(NP[dtype]), 5003
    host = [rng.integers(info.min, info.max, n, dtype=NP[dtype], endpoint=True) for _ in range(world)]
    host[0][:9], host[1][:9] = info.max, info.max
    dev = [torch.from_numpy(v).cuda() for v in host]
    out = torch.zeros_like(dev[0])
    torch.cuda.synchronize()
    code = DTYPE[dtype]
    assert H.ranks_sum([out.data_ptr()], [t.data_ptr() for t in dev], [n], world, code, code, code, 1.0, 1.0, gpu.stream)
    gpu.stream.synchronize()
    want = host[0].copy()
    for v in host[1:]:
        want += v  # numpy's arrays wrap
    assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("dtype", ["uint8", "int8"])
@pytest.mark.parametrize("world", [1, 2, 4, 9])
@pytest.mark.parametrize("pre,post", [(3.0, 1.0), (7.3, 0.5), (-1.0, 1.0), (1.0, 3.7), (5.0, 5.0)])
def test_scaled_bytes_beyond_their_range_wrap_like_the_oracle(gpu, orc, dtype, world, pre, post):
    """Every byte value, scaled to several times its range, and no trace of it in the bytes beside."""
    rng = np.random.default_rng(world)
    n = 5 * 256 + 3
    host = [rng.permutation(np.arange(n) % 256).astype(np.uint8).view(NP[dtype]) for _ in range(world)]
    dev = [torch.from_numpy(v).cuda() for v in host]
    out = torch.zeros_like(dev[0])
    torch.cuda.synchronize()
    code = DTYPE[dtype]
    assert H.ranks_sum([out.data_ptr()], [t.data_ptr() for t in dev], [n], world, code, code, code, pre, post, gpu.stream)
    gpu.stream.synchronize()
    assert np.array_equal(out.cpu().numpy(), _expected(orc, host, dtype, dtype, pre, post))


def test_ranks_sum_into_and_out_of_a_buffer(gpu, orc):
    """FLOAT32 tensors into a FLOAT16 fusion buffer, pad bytes zeroed, and out again."""
    rng = np.random.default_rng(3)
    counts = [5, 1024, 2049, 1]
    offs = np.cumsum([0] + [(2 * c + 15) // 16 * 16 for c in counts])
    a, b = ([rng.uniform(-2, 2, c).astype(np.float32) for c in counts] for _ in range(2))
    da, db = ([torch.from_numpy(v).cuda() for v in x] for x in (a, b))
    buf = torch.full((int(offs[-1]),), 255, dtype=torch.uint8, device="cuda")
    out = [torch.zeros_like(t) for t in da]
    torch.cuda.synchronize()
    f32, f16 = DTYPE["float32"], DTYPE["float16"]
    at = [buf.data_ptr() + int(o) for o in offs[:-1]]
    assert H.ranks_sum(at, [t.data_ptr() for t in da + db], counts, 2, f32, f16, f16, 0.25, 1.0, gpu.stream, pad=True)
    assert H.ranks_sum([t.data_ptr() for t in out], at, counts, 1, f16, f16, f32, 1.0, 3.0, gpu.stream)
    gpu.stream.synchronize()
    image = buf.cpu().numpy()
    for i, c in enumerate(counts):
        half = [v.astype(np.float16) for v in (a[i], b[i])]
        want = _expected(orc, half, "float16", "float16", 0.25, 1.0)
        piece = image[offs[i]:offs[i + 1]]
        assert np.array_equal(piece[:2 * c], want.view(np.uint8)) and not piece[2 * c:].any()
        got = out[i].cpu().numpy()
        assert np.array_equal(got, orc.scale_buffer(want, 3.0, f16).astype(np.float32))


def test_ranks_sum_refuses_overlap(gpu):
    t = torch.zeros(4096, dtype=torch.float32, device="cuda")
    p, f32 = t.data_ptr(), DTYPE["float32"]
    call = lambda outs, ins, counts, world: H.ranks_sum(outs, ins, counts, world, f32, f32, f32, 1.0, 1.0, gpu.stream)  # noqa: E731
    assert call([p, p + 400], [p, p + 400], [100, 100], 1)
    assert not call([p, p + 396], [p + 8192, p + 12000], [100, 100], 1)        # output over output
    assert not call([p], [p + 4], [100], 1)                                    # output over a shifted input
    assert not call([p, p + 400], [p, p + 400, p + 400, p], [100, 100], 2)     # output over another entry's input


# tensors that one launch carries, by the number of ranks
CARRIED = {1: 128, 2: 128, 3: 128, 5: 121, 8: 84, 9: 40}


@pytest.mark.parametrize("world", CARRIED)
@pytest.mark.parametrize("more", [-1, 0, 1, None])
def test_as_many_tensors_as_a_launch_carries_and_more(gpu, world, more):
    """Wherever they lie: each rank's tensors, and the outputs, in an order of their own within one allocation."""
    n = 2 * CARRIED[world] + 3 if more is None else CARRIED[world] + more
    rng = np.random.default_rng(n)
    counts = [int(x) for x in rng.choice([1, 3, 256, 1023, 1025], n)]

    def scattered():
        whole = torch.empty(1030 * n, dtype=torch.float32, device="cuda").normal_()
        return whole, [whole[1030 * int(k):1030 * int(k) + c] for k, c in zip(rng.permutation(n), counts)]

    ranks = [scattered() for _ in range(world)]
    whole, outs = scattered()
    want = whole.clone()
    for i, o in enumerate(outs):
        acc = ranks[0][1][i].clone()
        for r in range(1, world):
            acc += ranks[r][1][i]
        at = o.storage_offset()
        want[at:at + counts[i]] = acc
    torch.cuda.synchronize()
    f32 = DTYPE["float32"]
    assert H.ranks_sum([o.data_ptr() for o in outs], [t.data_ptr() for _, r in ranks for t in r], counts, world, f32, f32,
                       f32, 1.0, 1.0, gpu.stream)
    gpu.stream.synchronize()
    assert torch.equal(whole, want)


@pytest.mark.parametrize("world", [1, 2, 3, 8])
def test_tensors_that_32_bits_do_not_span(gpu, world):
    """Bytes more than 2^32 apart in one rank or in the outputs, and a tensor of more than 2^32 of them."""
    u8, far = DTYPE["uint8"], (1 << 32) + 70001
    big = [torch.empty(far, dtype=torch.uint8, device="cuda").random_() for _ in range(world)]
    out = torch.zeros(far + 16, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    assert H.ranks_sum([out.data_ptr()], [b.data_ptr() for b in big], [far], world, u8, u8, u8, 1.0, 1.0, gpu.stream)
    gpu.stream.synchronize()
    acc = big[0].clone()
    for b in big[1:]:
        acc += b
    assert torch.equal(out[:far], acc) and not out[far:].any()
    del acc
    # The first rank's tensors at both ends in turn, the others' close together; then the outputs.  As few as two, more
    # than a launch carries with such distances, and close ones ahead of the first that is far.
    n = 5000
    for count, close in ((3, 0), (200, 0), (200, 70)):
        at = [i * n if i % 2 == 0 or i < close else far - (i + 1) * n for i in range(count)]
        near = [[torch.empty(n, dtype=torch.uint8, device="cuda").random_() for _ in at] for _ in range(world)]
        spread, small = [out[a:a + n] for a in at], [torch.empty(n, dtype=torch.uint8, device="cuda") for _ in at]
        torch.cuda.synchronize()
        for outs, first in ((small, [big[0][a:a + n] for a in at]), (spread, near[0])):
            ranks = [first] + near[1:]
            assert H.ranks_sum([o.data_ptr() for o in outs], [t.data_ptr() for r in ranks for t in r], [n] * count, world,
                               u8, u8, u8, 1.0, 1.0, gpu.stream)
            gpu.stream.synchronize()
            for i, o in enumerate(outs):
                acc = ranks[0][i].clone()
                for r in ranks[1:]:
                    acc += r[i]
                assert torch.equal(o, acc), (count, i)


@pytest.mark.parametrize("case", ["peers_are_outputs", "same_output_twice", "more_ranks_than_one_pass"])
def test_engine_sums_through_a_buffer_where_one_pass_cannot(monkeypatch, case):
    import horovod_amd.torch as hvd
    hvd.shutdown()
    size = 5 if case == "more_ranks_than_one_pass" else 2
    x, y = (torch.arange(n, dtype=torch.float32, device="cuda") + n for n in (1000, 1000))
    xs, ys = x.cpu(), y.cpu()
    if case == "more_ranks_than_one_pass":
        monkeypatch.setattr(H, "RANKS_SUM_MAX_WORLD", 2)
    # rank 1 passes the other entry's tensor, which is overwritten in place
    hvd.init(size=size, peer_source=(lambda r, name, t: y if t is x else x) if case == "peers_are_outputs" else None)
    try:
        if case == "same_output_twice":
            y, ys = x, xs
        handles = [hvd.allreduce_async_(t, op=hvd.Sum) for t in (x, y)]
        for h in handles:
            hvd.synchronize(h)
        if case == "peers_are_outputs":
            assert torch.equal(x.cpu(), xs + ys) and torch.equal(y.cpu(), xs + ys)
        else:
            assert torch.equal(x.cpu(), size * xs) and torch.equal(y.cpu(), size * ys)
    finally:
        hvd.shutdown()


def test_a_response_that_fails_halfway_waits_for_what_it_queued(monkeypatch):
    """Adasum over two nodes of four ranks, and no buffer for the second node's sum: the first one's is under way
    and reads tensors that the caller is free to drop once it has the error."""
    import horovod_amd.torch as hvd
    from horovod_amd.torch import mpi_ops
    hvd.shutdown()
    hvd.init(size=8, local_size=4)
    engine = mpi_ops._engine
    buffer = engine._buffer

    def no_second_node(slot, what, nbytes):
        if what == 3:
            raise MemoryError("no second buffer")
        return buffer(slot, what, nbytes)

    try:
        t = torch.zeros(1 << 29, dtype=torch.float32, device="cuda")
        stream = torch.cuda.ExternalStream(engine.streams[0].handle.value)
        engine._buffer(0, 2, t.numel() * 4)
        torch.cuda.synchronize()
        monkeypatch.setattr(engine, "_buffer", no_second_node)
        handle = hvd.allreduce_async(t, op=hvd.Adasum)
        engine.run_cycle()
        assert stream.query()  # 2 GiB: more than a millisecond of work
        with pytest.raises(hvd.HorovodInternalError, match="no second buffer"):
            hvd.synchronize(handle)
        monkeypatch.undo()
        assert torch.equal(hvd.allreduce(t[:1000], op=hvd.Adasum), t[:1000])
    finally:
        hvd.shutdown()
