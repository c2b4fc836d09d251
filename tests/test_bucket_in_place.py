"""DiLoCo's bucketised all-reduce with kernels that work on the tensors in place, against the same
step by way of copies into and out of the flat buffer, by bytes."""

import time

import pytest
import torch
from torch.distributed import ReduceOp

import sim_pg
from sim_pg import SimGroup
from test_gpu_collectives import run_ranks
from torchft_amd import allreduce as ar


def refused(kind, t):
    """`t` as a tensor that only a copy can take, and the piece of a flat buffer it belongs to"""
    piece = torch.zeros(t.numel()).view_as(t)
    if kind == "strided":
        return t.t().contiguous().t(), piece
    if kind == "dtype":
        return t.to(torch.bfloat16), piece
    if kind == "autograd":
        return t.requires_grad_(), piece
    if kind == "shape":
        return t[:1], piece
    if kind == "subclass":
        return t.as_subclass(type("Other", (torch.Tensor,), {})), piece
    if kind == "negated":
        return torch._neg_view(t), piece
    return t, piece


@pytest.mark.parametrize("kind", ["strided", "dtype", "autograd", "shape", "subclass", "negated", "plain"])
def test_what_only_a_copy_can_take(kind):
    plain = torch.ones(3, 4)
    t, piece = refused(kind, torch.ones(3, 4))
    got = ar._addresses([plain, t], [torch.zeros(3, 4), piece])
    assert got == ([plain.data_ptr(), t.data_ptr()] if kind == "plain" else None)
    with torch.autograd.forward_ad.dual_level():
        assert ar._addresses([plain], [torch.zeros(3, 4)]) is None


def test_what_functorch_follows():
    plain, piece = torch.ones(3, 4), torch.zeros(3, 4)
    seen = []

    def look(t):
        seen.append(ar._addresses([t], [piece]))
        return t.sum()

    torch.func.grad(look)(plain)
    torch.func.vmap(look)(plain.expand(2, 3, 4).contiguous())
    torch.func.functionalize(look)(plain)
    with torch.inference_mode():
        seen.append(ar._addresses([torch.ones(3, 4)], [piece]))
    meta = torch.empty(3, 4, device="meta")
    seen.append(ar._addresses([meta], [meta]))
    seen.append(ar._addresses([torch._efficientzerotensor((3, 4))], [piece]))
    assert seen == [None] * 6


def test_addresses_that_are_known():
    tensors = [torch.empty(i % 4, 5) for i in range(50)]
    pieces = [torch.empty_like(t) for t in tensors]
    known = ar._addresses(tensors, pieces)
    assert known == [t.data_ptr() for t in tensors]
    assert ar._addresses(tensors, pieces, known) is known
    tensors[9].data = torch.empty(1, 5)
    moved = ar._addresses(tensors, pieces, known)
    assert moved == [t.data_ptr() for t in tensors] and moved is not known
    assert ar._addresses(tensors, pieces, known[:-1]) == moved
    base = torch.empty(40)
    for parts, shared in (([base[:10], base[10:20], base[30:40], base[20:30]], False), ([base[:11], base[10:20]], True),
                          ([base[5:10], base[0:40]], True), ([base[5:5], base[0:40]], False), ([base, base], True)):
        pieces = [torch.empty_like(t) for t in parts]
        assert ar._addresses(parts, pieces) == (None if shared else [t.data_ptr() for t in parts])


def test_host_time_per_tensor():
    """What a step does per tensor besides its launches (the copies cost 0.25 us per tensor and way)."""
    tensors = [torch.empty(3, 5) for _ in range(2000)]
    pieces = [torch.empty_like(t) for t in tensors]
    known = ar._addresses(tensors, pieces)
    times = []
    for _ in range(20):
        begin = time.perf_counter()
        assert ar._addresses(tensors, pieces, known) is known
        times.append(time.perf_counter() - begin)
    assert min(times) < 2000 * 0.3e-6


def step(peers, ws, dtype, capacity, op, way, monkeypatch, aliased=False):
    """Two steps on copies of the peers' tensors; what every rank holds after each, and the buckets.
    `aliased`: in the first step two tensors of one storage"""
    group, seen = SimGroup(ws), [[] for _ in range(ws)]
    mine = [[t.cuda() for t in tensors] for tensors in peers]
    if way == "copies":
        monkeypatch.setattr(ar.BucketizedAllreduce, "_in_place", lambda self, bucket, whole: None)
    if aliased:
        for tensors in mine:
            tensors[2] = tensors[3][:tensors[2].numel()].view_as(tensors[2])
    averaging = [ar.BucketizedAllreduce(tensors, capacity * tensors[0].element_size()) for tensors in mine]
    for a in averaging:
        a.made = []  # after each step: the buckets in place that exist

    def rank_fn(r):
        for _ in range(2):
            works = averaging[r].allreduce(group.rank(r), ws, reduce_op=op)
            assert all(w.wait() and w.get_future().value() == [] for w in works)
            seen[r].append([t.clone() for t in mine[r]])
            averaging[r].made.append([len(b["piecewise"]) for b in averaging[r].buckets])
            for t in mine[r]:
                t.data = t * 0.5  # storage of its own for the second step

    run_ranks(ws, rank_fn, group)
    torch.cuda.synchronize()
    monkeypatch.undo()
    return seen, averaging


@pytest.mark.gpu
@pytest.mark.parametrize("op", [ReduceOp.SUM, ReduceOp.AVG])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ws,sizes,capacity", [
    (2, [(64, 48), (1,), (7, 33), (2049,), (0,), (3, 1)], 1 << 20),   # one buffer; odd starts
    (3, [(2047,), (5, 5), (1, 1), (4096, 3)], 1 << 20),               # padding rows
    (4, [(6,), (6,), (6,), (6,)], 8),                                 # buffers with a rest that no tensor covers
    (5, [(k % 7 + 1, 2 * k + 1) for k in range(40)], 1 << 20),        # addresses that travel through device memory
    (1, [(1025,)], 1 << 20),
])
def test_in_place_step_has_the_bytes_of_the_copies(monkeypatch, dtype, ws, sizes, capacity, op):
    g = torch.Generator().manual_seed(len(sizes))
    peers = [[(torch.randn(s, generator=g) * 0.1).to(dtype) for s in sizes] for _ in range(ws)]
    got, averaging = step(peers, ws, dtype, capacity, op, "in place", monkeypatch)
    assert all(b["piecewise"] for a in averaging for b in a.buckets if b["owners"])
    want, averaging = step(peers, ws, dtype, capacity, op, "copies", monkeypatch)
    assert not any(b["piecewise"] for a in averaging for b in a.buckets)
    for r in range(ws):
        for k in range(2):
            for i, (a, b) in enumerate(zip(got[r][k], want[r][k])):
                assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8)), (r, k, sizes[i])


@pytest.mark.gpu
def test_shared_memory_and_storage_that_moves_in_flight(monkeypatch):
    g = torch.Generator().manual_seed(3)
    peers = [[torch.randn(s, generator=g) for s in [(16,), (9, 9), (5, 4), (300,)]] for _ in range(2)]
    got, averaging = step(peers, 2, torch.float32, 1 << 20, ReduceOp.AVG, "in place", monkeypatch, aliased=True)
    # the first step has shared memory and copies; afterwards every tensor has storage of its own
    assert all(a.made == [[0], [1]] for a in averaging)
    want, _ = step(peers, 2, torch.float32, 1 << 20, ReduceOp.AVG, "copies", monkeypatch, aliased=True)
    assert all(torch.equal(a, b) for r in range(2) for k in range(2) for a, b in zip(got[r][k], want[r][k]))

    want, _ = step(peers, 2, torch.float32, 1 << 20, ReduceOp.AVG, "copies", monkeypatch)
    group = SimGroup(2)
    mine = [[t.cuda() for t in tensors] for tensors in peers]
    versions = [[t._version for t in tensors] for tensors in mine]
    gather = type(group.rank(0)).allgather_into_tensor_coalesced

    def moving(self, *args, **kwargs):
        mine[self.rank()][1].data = torch.zeros(9, 9, device="cuda")
        return gather(self, *args, **kwargs)

    monkeypatch.setattr(type(group.rank(0)), "allgather_into_tensor_coalesced", moving)
    averaging = [ar.BucketizedAllreduce(tensors, 1 << 20) for tensors in mine]

    def rank_fn(r):
        for w in averaging[r].allreduce(group.rank(r), 2):
            w.wait()

    run_ranks(2, rank_fn, group)
    torch.cuda.synchronize()
    for r in range(2):
        assert all(torch.equal(a, b) for a, b in zip(mine[r], want[r][0]))
        assert all(t._version > v for i, (t, v) in enumerate(zip(mine[r], versions[r])) if i != 1)


class Whole:
    """Stands for the prepared bucket of the flat buffer."""
    ws, device = 2, torch.device("cpu")


@pytest.mark.parametrize("count,capacity", [(16, 64), (15, 61), (16, 61), (17, 68), (40, 1 << 10)])
def test_no_table_is_made_under_a_capture(monkeypatch, count, capacity):
    # capacity 64 + or - 3 of tensors of 4 elements: with or without a rest that no tensor covers
    tensors = [torch.ones(4) for _ in range(count)]
    averaging = ar.BucketizedAllreduce(tensors, 4 * capacity)
    bucket = averaging.buckets[0]
    parts = len(bucket["owners"]) + (bucket["used"] < bucket["flat"].numel())
    capturing = [True]
    monkeypatch.setattr(ar._q, "_capturing", lambda device: capturing[0])
    monkeypatch.setattr(ar._q, "PreparedBucket", lambda plan, *rest: plan)
    made = averaging._in_place(bucket, Whole)
    assert (made is None) == (parts > 16)
    if made is not None:
        assert made._parts.n_tensors == parts and bucket["captured"] == [made]
        return
    assert not bucket["piecewise"] and not bucket["captured"]
    capturing[0] = False
    made = averaging._in_place(bucket, Whole)   # an eager step makes the table ...
    assert made._parts.n_tensors == parts and not bucket["captured"]
    capturing[0] = True
    assert averaging._in_place(bucket, Whole) is made and bucket["captured"] == [made]   # ... for captures after it
    bucket["owners"][3].data = torch.ones(4)
    assert averaging._in_place(bucket, Whole) is None


class OneRank:
    """Rank 0 of a group whose other ranks send what `others` holds."""

    def __init__(self, others):
        self.others = others

    def rank(self):
        return 0

    def size(self):
        return len(self.others)

    def alltoall_base(self, output, input, output_splits, input_splits, opts=None):
        output.copy_(self.others)
        output[0].copy_(input[0])
        return sim_pg._DoneWork()

    def allgather_into_tensor_coalesced(self, outputs, inputs, opts=None):
        outputs[0].copy_(self.others)
        outputs[0][:1].copy_(inputs[0])
        return sim_pg._DoneWork()


@pytest.mark.gpu
@pytest.mark.parametrize("count", [9, 40])
@pytest.mark.parametrize("warm", [False, True])
def test_a_step_under_a_capture(count, warm):
    """The graph replayed between eager steps, each against the same step by way of the copies."""
    g = torch.Generator().manual_seed(count)
    start = [torch.randn(3 * i % 50 + 1, 5, generator=g) for i in range(count)]
    total = sum(t.numel() for t in start)
    peer = ar._q.fused_quantize_into_fp8([torch.randn(total, generator=g).cuda()], 2).view(2, -1)
    want = [t.cuda() for t in start]
    copies = ar.BucketizedAllreduce(want, 4 * total)
    copies._in_place = lambda bucket, whole: None
    mine = [t.cuda() for t in start]
    averaging = ar.BucketizedAllreduce(mine, 4 * total)

    def step(averaging):
        for w in averaging.allreduce(OneRank(peer), 2):
            w.wait()

    def check(what):
        torch.cuda.synchronize()
        for a, b in zip(mine, want):
            assert torch.equal(a, b), what

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        if warm:
            step(averaging)
            step(copies)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step(averaging)
        assert bool(averaging.buckets[0]["captured"]) == (warm or count <= 16)
        check("the capture itself")
        step(averaging)   # eager, on the stream of the capture, before the first replay
        step(copies)
        check("eager step behind the capture")
        for k in range(3):
            for t, w in zip(mine, want):
                t.mul_(1.5)
                w.mul_(1.5)
            graph.replay()
            step(copies)
            check(f"replay {k}")
            step(averaging)
            step(copies)
            check(f"eager step {k}")
