"""Lists on both sides of the length from which their addresses reach the device by a copy from
pinned memory: new addresses on every call, on several streams, named functions and buckets."""

import contextlib
import threading

import pytest
import torch

from torchft_amd import quantization as q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [17, q._COPY_FROM - 1, q._COPY_FROM, 2500])
def test_addresses_of_every_call_arrive(n):
    g = torch.Generator().manual_seed(n)
    lists = [[torch.randn(3, 9, generator=g).cuda() for _ in range(n)] for _ in range(3)]
    # the same bytes by way of one [3 n, 9] matrix in a group of one
    want = [q.fused_quantize_into_fp8([torch.cat(ts)], 1) for ts in lists]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for k in range(12):
        with torch.cuda.stream(streams[k % 2]):
            if k < 9:
                got.append((k % 3, q.fused_quantize_into_fp8(list(lists[k % 3]), 1)))
            else:
                got.append((k % 3, q.prepare(list(lists[k % 3]), 1).quantize()))
    torch.cuda.synchronize()
    assert all(torch.equal(packed, want[i]) for i, packed in got)
    out = [torch.zeros_like(t) for t in lists[0]]
    q.fused_dequantize_from_fp8(out, want[1], 1)
    q.fused_dequantize_from_fp8(lists[1], want[1], 1)
    assert all(torch.equal(a, b) for a, b in zip(out, lists[1]))


@pytest.mark.parametrize("n", [q._COPY_FROM - 1, q._COPY_FROM])
@pytest.mark.parametrize("way", ["functions", "bucket"])
@pytest.mark.parametrize("first,then", [("inference", "plain"), ("plain", "inference"), ("inference", "inference"),
                                        ("cuda", "plain"), ("plain", "cuda"), ("meta", "plain"), ("plain", "meta")])
def test_addresses_in_other_modes(n, way, first, then):
    """Calls inside and outside of inference mode, and with another default device, on new addresses."""
    modes = {"plain": contextlib.nullcontext, "inference": torch.inference_mode,
             "cuda": lambda: torch.device("cuda"), "meta": lambda: torch.device("meta")}
    cols = 11 + len(first) + 20 * len(then) + 100 * (way == "bucket")  # a plan of its own for every case
    g = torch.Generator().manual_seed(n)
    lists = [[torch.randn(2, cols, generator=g).cuda() for _ in range(n)] for _ in range(3)]
    want = [q.fused_quantize_into_fp8([torch.cat(ts)], 1) for ts in lists]
    made = {}
    for k, mode in enumerate([first, then, first]):
        with modes[mode]():
            if way == "bucket":   # made in one mode, first used in the other
                made[k] = q.prepare(lists[k], 1)
                with modes["plain" if mode != "plain" else then]():
                    got = made[k].quantize()
            else:
                got = q.fused_quantize_into_fp8(lists[k], 1)
        assert torch.equal(got, want[k]), (k, mode)


@pytest.mark.parametrize("side", [False, True])
@pytest.mark.parametrize("n", [q._COPY_FROM - 1, q._COPY_FROM, 9000])
def test_new_addresses_while_another_thread_captures(n, side):
    """A capture in global mode, and calls of this thread meanwhile with new addresses every time,
    more of them than the pinned allocator has memory of that size for."""
    g = torch.Generator().manual_seed(n)
    lists = [[torch.randn(2, 5, generator=g).cuda() for _ in range(n)] for _ in range(6)]
    want = [q.fused_quantize_into_fp8([torch.cat(ts)], 1) for ts in lists]
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    with torch.cuda.stream(stream):
        q.fused_quantize_into_fp8(lists[0], 1)   # the plan's table and this stream's buffer
        buckets = [q.prepare(ts, 1) for ts in lists]
        outs = [torch.empty_like(w) for w in want]
        # what the calls below allocate: torch may not ask for more then, and gives back whole segments before
        spare = [torch.empty_like(w) for w in want for _ in range(3)]
        del spare[::2]
    torch.cuda.synchronize()
    x = torch.arange(1024, device="cuda", dtype=torch.float32)
    y = torch.zeros_like(x)
    torch.cuda.synchronize()
    graph, began, finish, failed = torch.cuda.CUDAGraph(), threading.Event(), threading.Event(), []

    def capture():
        try:
            with torch.cuda.graph(graph, capture_error_mode="global"):
                y.copy_(x * 2)
                began.set()
                finish.wait(60)
                y.add_(1)
        except Exception as e:  # reported below
            failed.append(e)
            began.set()

    thread = threading.Thread(target=capture)
    thread.start()
    began.wait(60)
    got = []
    try:
        with torch.cuda.stream(stream):
            for ts, bucket, out in zip(lists, buckets, outs):
                got.append(q.fused_quantize_into_fp8(ts, 1))
                got.append(bucket.quantize(out))
    finally:
        finish.set()
        thread.join()
    assert not failed, failed
    torch.cuda.synchronize()
    assert all(torch.equal(packed, want[k // 2]) for k, packed in enumerate(got))
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, x * 2 + 1)
