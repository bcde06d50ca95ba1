"""hvdhip_adasum_ranks against the oracle's pairwise combine, level by level, at the edges of its chunks (16 KiB of
the wire type), of the partial sums that a consumer adds itself (512 per tensor; "long" at 8 and 16 ranks has every
level read the coefficients of the launch in between), of the tensors one launch carries (77 of eight ranks), of the
ranks one launch reads (8) and of what the first pass leaves in the Infinity Cache (all ranks up to 160 MiB in
total, of 16 "long" ones every other)."""
import numpy as np
import pytest
import torch

from horovod_amd import DTYPE
from horovod_amd import host as H

pytestmark = pytest.mark.gpu

NP = {"float16": np.float16, "float32": np.float32, "float64": np.float64}


def _tree(orc, ranks, wire, pre, post):
    code = DTYPE[wire]
    level = [v.astype(NP[wire]) for v in ranks]
    level = [orc.scale_buffer(v, pre, code) if pre != 1.0 else v for v in level]
    while len(level) > 1:
        level = [orc.adasum_pairwise(a, b, [a.size], code)[0] for a, b in zip(level[::2], level[1::2])]
    return orc.scale_buffer(level[0], post, code) if post != 1.0 else level[0]


@pytest.mark.parametrize("dtype,wire", [(d, d) for d in NP] + [("float32", "float16")])
@pytest.mark.parametrize("world,shape", [(2, "edges"), (4, "edges"), (8, "edges"), (32, "edges"), (64, "edges"),
                                         (128, "edges"), (4, "long"), (8, "long"), (16, "long"), (8, "rows")])
def test_adasum_ranks_equals_the_pairwise_tree(gpu, orc, dtype, wire, world, shape):
    rng = np.random.default_rng(world)
    chunk = 16384 // np.dtype(NP[wire]).itemsize
    counts = {"edges": [1, 0, 3, chunk - 1, chunk, chunk + 1, 2 * chunk + 7, 255],
              "long": [5, 512 * chunk, 512 * chunk + 1, 0],
              "rows": [int(x) for x in rng.integers(0, 300, 100)]}[shape]
    pre, post = (0.125, 0.3) if world % 8 else (1.0, 1.0)
    host = [[rng.normal(0.0, 0.01 * (1 + r), c).astype(NP[dtype]) for c in counts] for r in range(world)]
    # one element into the allocation each: only element alignment is promised
    dev = [[torch.from_numpy(np.concatenate([v[:1], v])).cuda()[1 if v.size else 0:] for v in rank] for rank in host]
    out = [torch.zeros(c + 1, dtype=dev[0][0].dtype, device="cuda") for c in counts]
    code, wcode = DTYPE[dtype], DTYPE[wire]
    need = H.adasum_ranks_workspace(counts, world, wcode)
    work = torch.full((need + 256,), 255, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    flat = [t.data_ptr() for r in dev for t in r]
    for to in ([o.data_ptr() for o in out], [t.data_ptr() for t in dev[0]]):  # and in place: rank 0's tensors
        assert H.adasum_ranks(to, flat, counts, world, code, wcode, code, pre, post, work.data_ptr(), need, gpu.stream)
    gpu.stream.synchronize()
    assert bool((work[need:] == 255).all()), "wrote behind the workspace"
    levels = world.bit_length() - 1
    for i, c in enumerate(counts):
        if c == 0:
            continue
        ranks = [host[r][i] for r in range(world)]
        want = _tree(orc, ranks, wire, pre, post).astype(np.float64)
        got = out[i].cpu().numpy()
        assert got[c] == 0, "wrote behind its tensor"
        assert np.array_equal(got[:c].view(np.uint8), dev[0][i].cpu().numpy().view(np.uint8)), (i, c)
        diff = np.abs(got[:c].astype(np.float64) - want)
        # The oracle adds the c products of a sum one after the other: off by up to c units of 2^-53 of |a||b|, which
        # moves a coefficient (at most 1.5) by half of that; a rounding to the wire type that tips moves by an ulp.
        # Both scale with the ranks' magnitudes, which a level multiplies by at most 1.5.
        size = sum(np.abs(v.astype(np.float64)) for v in ranks) * 1.5 ** levels * pre * post
        ulp = {"float16": 2.0 ** -10, "float32": 2.0 ** -23, "float64": 2.0 ** -52}[wire]
        assert (diff <= levels * (ulp + (c + 64) * 2.0 ** -53) * size + 2.0 ** -24).all(), (i, c, diff.max())
        if wire != "float64":  # a tipped rounding needs a value within about 1e-13 of a midpoint
            assert np.count_nonzero(diff) <= 2 + 1e-5 * c, (i, c, np.count_nonzero(diff))


@pytest.mark.parametrize("world", [2, 8, 16])
def test_adasum_ranks_does_not_depend_on_the_other_tensors(gpu, world):
    """A tensor of up to 512 chunks gives the same bits by itself and beside one of more, where the coefficients of
    all come from a launch of their own.  In float64, with ranks that have much in common, a coefficient's last bit
    shows in most elements, and sums in another order move it in some pair of some tensor."""
    gen = torch.Generator(device="cuda").manual_seed(world)
    chunk, code = 16384 // 8, DTYPE["float64"]
    counts = [130 * chunk + 5 * i for i in range(6)] + [300 * chunk + 17, 512 * chunk, 513 * chunk]

    def normal(c):
        return torch.empty(c, dtype=torch.float64, device="cuda").normal_(0.0, 0.01, generator=gen)

    common = [normal(c) for c in counts]
    dev = [[t + normal(t.numel()) for t in common] for _ in range(world)]

    def combine(which):
        sizes = [counts[i] for i in which]
        out = [torch.zeros(c, dtype=torch.float64, device="cuda") for c in sizes]
        need = H.adasum_ranks_workspace(sizes, world, code)
        work = torch.empty(need, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        assert H.adasum_ranks([o.data_ptr() for o in out], [r[i].data_ptr() for r in dev for i in which], sizes, world,
                              code, code, code, 1.0, 1.0, work.data_ptr(), need, gpu.stream)
        gpu.stream.synchronize()
        return out

    together = combine(range(len(counts)))
    for i in range(len(counts)):
        assert torch.equal(combine([i])[0].view(torch.int64), together[i].view(torch.int64)), counts[i]


@pytest.mark.parametrize("dtype", NP)
@pytest.mark.parametrize("world", [2, 4, 8])
@pytest.mark.parametrize("chunks", [1, 2])
@pytest.mark.parametrize("scaled", [False, True])
def test_short_rows_give_the_same_bits_in_one_launch(gpu, dtype, world, chunks, scaled):
    """Rows of up to two chunks go through the tree in one launch when all of a response's are so short; beside a row of
    three chunks they go level by level.  Rows at the ends of vectors and chunks, one element into their allocations;
    more rows than a launch carries; sums that are not finite; ranks that cancel."""
    es = np.dtype(NP[dtype]).itemsize
    chunk, code = 16384 // es, DTYPE[dtype]
    counts = [1, 0, 16 // es - 1, 255 * 16 // es, 3 * 4096 // es + 5, chunk - 1, chunk, 7]
    if chunks == 2:
        counts += [chunk + 1, 2 * chunk - 1, 2 * chunk, chunk + 16 // es]
    counts += [33 + i for i in range(100)]  # more than a launch carries; the long row below comes first of all
    gen = torch.Generator(device="cuda").manual_seed(world)
    kind = getattr(torch, dtype)

    def draw(n):
        return torch.empty(n + 1, dtype=kind, device="cuda").normal_(0.0, 0.1, generator=gen)

    long_row = 2 * chunk + 1
    base = [draw(n) for n in counts]
    ranks = [[b * 0.5 + draw(n) for b, n in zip(base, counts)] for _ in range(world)]
    longs = [draw(long_row) for _ in range(world)]
    ranks[1][7][:] = -ranks[0][7]                     # a pair that cancels
    ranks[0][5][3], ranks[1][6][2] = float("nan"), float("inf")
    pre, post = (0.3, 1.7) if scaled else (1.0, 1.0)

    def run(beside_a_long_row, in_place):
        sizes = [long_row] * beside_a_long_row + counts
        ins = [[t.clone() for t in [row] * beside_a_long_row + r] for row, r in zip(longs, ranks)]
        outs = ins[0] if in_place else [torch.zeros_like(t) for t in ins[0]]
        need = H.adasum_ranks_workspace(sizes, world, code)
        work = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        assert H.adasum_ranks([t.data_ptr() + es for t in outs], [t.data_ptr() + es for r in ins for t in r], sizes, world,
                              code, code, code, pre, post, work.data_ptr(), need, gpu.stream)
        gpu.stream.synchronize()
        return outs[beside_a_long_row:]

    alone, in_place, general = run(False, False), run(False, True), run(True, False)
    for i, n in enumerate(counts):
        want = general[i].view(torch.uint8)
        assert torch.equal(alone[i].view(torch.uint8), want), (i, n)
        assert torch.equal(in_place[i][1:].view(torch.uint8), want[es:]), (i, n)
        assert torch.equal(in_place[i][:1].view(torch.uint8), ranks[0][i][:1].view(torch.uint8)), (i, n)


@pytest.mark.parametrize("world", [2, 8])
@pytest.mark.parametrize("count,n", [(3, 3 * 8192 + 5), (100, 3 * 8192 + 5), (100, 1000)])
def test_rows_that_32_bits_do_not_span(gpu, world, count, n):
    """Halves more than 2^32 elements apart in turn, in a rank and then in the outputs: the bits that the rows give close
    together.  More rows than a launch carries with such distances, through the levels and in one launch."""
    code, far = DTYPE["float16"], 1 << 32
    gen = torch.Generator(device="cuda").manual_seed(world)
    wide = torch.empty(far + count * n, dtype=torch.float16, device="cuda")
    ends = [wide[i * n:(i + 1) * n] if i % 2 else wide[far + i * n:far + (i + 1) * n] for i in range(count)]
    ranks = [[torch.empty(n, dtype=torch.float16, device="cuda").normal_(generator=gen) for _ in ends] for _ in range(world)]
    need = H.adasum_ranks_workspace([n] * count, world, code)
    work = torch.empty(need, dtype=torch.uint8, device="cuda")

    def run(outs, ins):
        torch.cuda.synchronize()
        assert H.adasum_ranks([o.data_ptr() for o in outs], [t.data_ptr() for r in ins for t in r], [n] * count, world, code,
                              code, code, 1.0, 1.0, work.data_ptr(), need, gpu.stream)
        gpu.stream.synchronize()
        return [o.clone() for o in outs]

    want = run([torch.zeros_like(t) for t in ranks[0]], ranks)
    for e, t in zip(ends, ranks[1]):
        e.copy_(t)
    for got in (run([torch.zeros_like(t) for t in ranks[0]], ranks[:1] + [ends] + ranks[2:]), run(ends, ranks)):
        for g, w in zip(got, want):
            assert torch.equal(g.view(torch.int16), w.view(torch.int16))


def test_adasum_ranks_refuses(gpu):
    t = torch.zeros(8192, dtype=torch.float32, device="cuda")
    work = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    p, f32 = t.data_ptr(), DTYPE["float32"]

    def call(outs, ins, counts, world, space, dtype=f32):
        return H.adasum_ranks(outs, ins, counts, world, dtype, dtype, dtype, 1.0, 1.0, work.data_ptr(), space, gpu.stream)

    need = H.adasum_ranks_workspace([100, 100], 2, f32)
    assert call([p, p + 400], [p, p + 400, p + 8192, p + 8592], [100, 100], 2, need)
    assert not call([p, p + 396], [p + 8192, p + 8592] * 2, [100, 100], 2, need)  # output over output
    assert not call([p], [p + 4, p + 8192], [100], 2, need)                        # output over a shifted input
    for args in (([p], [p] * 3, [100], 3, 1 << 16), ([p], [p] * 2, [100], 2, 16), ([p], [p] * 2, [100], 2, 1 << 16, DTYPE["int32"])):
        with pytest.raises(Exception):
            call(*args)
    gpu.stream.synchronize()
