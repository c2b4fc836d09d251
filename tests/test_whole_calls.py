"""The named functions and prepared buckets on short lists whose plan is known: the call that
_pylist makes as a whole, and what it leaves to Python."""

import numpy as np
import pytest
import torch
from torch.distributed import ReduceOp
from torch.overrides import TorchFunctionMode

import torchft_amd
from torchft_amd import quantization as q


def test_host_tensors_are_left_to_python():
    if q._pylist is None:
        pytest.skip("torchft_amd._pylist cannot be built here")
    ts = [torch.zeros(4, 8)]
    packed = torch.zeros(8, dtype=torch.uint8)
    assert q._pylist.quantize(ts, 16, 2, {}) is None
    assert q._pylist.reduce(ts, 16, 2, {}, packed, 0, 1) is None
    assert q._pylist.dequantize(ts, 16, 2, {}, packed, None) is None
    assert q._pylist.quantize([torch.zeros(3)], 16, 2, {}) is None and q._pylist.quantize([], 16, 2, {}) is None
    with pytest.raises(TypeError):
        q._pylist.quantize(ts)


@pytest.fixture
def known(monkeypatch):
    """A list, a buffer of it, and a switch that makes any way through Python an error."""
    if q._pylist is None:
        pytest.skip("torchft_amd._pylist is not built")
    g = torch.Generator("cuda").manual_seed(3)
    ts = [torch.randn(33, 130, generator=g, device="cuda"), torch.randn(7, 1, generator=g, device="cuda")]
    packed = torchft_amd.fused_quantize_into_fp8(ts, 3)

    def only_whole_calls():
        def refuse(*_):
            raise AssertionError("not a whole call")
        monkeypatch.setattr(q, "_match_short_list", refuse)
        monkeypatch.setattr(q, "_check_packed", refuse)

    return ts, packed, only_whole_calls


@pytest.mark.gpu
@pytest.mark.parametrize("op", [ReduceOp.SUM, ReduceOp.AVG, ReduceOp(ReduceOp.SUM), ReduceOp.MAX])
def test_same_bytes_as_by_way_of_python(known, op, monkeypatch):
    ts, _, only_whole_calls = known
    want, got = [], []
    for out in (want, got):
        if out is got:
            only_whole_calls()
        else:
            monkeypatch.setattr(q, "_calls", None)
        copies = [t.clone() for t in ts]
        bucket = torchft_amd.prepare(copies, 3)
        packed = torchft_amd.fused_quantize_into_fp8(copies, 3)
        out += [packed.clone(), bucket.quantize()]
        for reduce in (lambda: torchft_amd.fused_reduce_fp8(copies, packed, 3, 1, op), lambda: bucket.reduce(packed, 2, op)):
            reduce()
            out.append(packed.clone())
        for dequantize in (lambda **k: torchft_amd.fused_dequantize_from_fp8(copies, packed, 3, **k),
                           lambda **k: bucket.dequantize(packed, **k)):
            for k in ({}, {"divide_by": 3}):
                dequantize(**k)
                out += [t.clone() for t in copies]
        monkeypatch.undo()
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
def test_what_is_wrong_is_said_as_before(known):
    ts, packed, _ = known
    bucket = torchft_amd.prepare(ts, 3)
    for reduce, dequantize in ((lambda p, r=0: torchft_amd.fused_reduce_fp8(ts, p, 3, r), lambda p: torchft_amd.fused_dequantize_from_fp8(ts, p, 3)),
                               (lambda p, r=0: bucket.reduce(p, r), lambda p: bucket.dequantize(p))):
        for call in (reduce, dequantize):
            with pytest.raises(AssertionError, match="Output size does not match"):
                call(packed[:-4])
            with pytest.raises(RuntimeError, match="contiguous uint8"):
                call(torch.empty(2 * packed.numel(), dtype=torch.uint8, device="cuda")[::2])
            with pytest.raises(RuntimeError, match="contiguous uint8"):
                call(packed.view(torch.int8))
            with pytest.raises(RuntimeError, match="the tensors are on"):
                call(packed.cpu())
        for rank in (-1, 3):
            with pytest.raises(RuntimeError, match="invalid argument"):
                reduce(packed, rank)
        a, b = packed.clone(), packed.clone()
        reduce(a, np.int64(2))  # any number that int() takes
        reduce(b, 2)
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_modes_see_the_allocation(known):
    ts, packed, _ = known
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        again = torchft_amd.fused_quantize_into_fp8(ts, 3)
    assert torch.empty in seen and torch.equal(again, packed)


@pytest.mark.gpu
def test_current_stream_and_capture(known):
    ts, packed, only_whole_calls = known
    only_whole_calls()
    side, out = torch.cuda.Stream(), torch.zeros_like(packed)
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        first = torchft_amd.fused_quantize_into_fp8(ts, 3)
        assert not side.query()  # behind what the stream is busy with
    side.synchronize()
    assert torch.equal(first, packed)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out.copy_(torchft_amd.fused_quantize_into_fp8(ts, 3))
        torchft_amd.fused_dequantize_from_fp8(ts, out, 3)
    want = None
    for _ in range(3):
        ts[0].add_(1.0)
        want = torchft_amd.fused_quantize_into_fp8(ts, 3)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
