"""Lists on both sides of the length from which their addresses reach the device by a copy from
pinned memory: new addresses on every call, on several streams, named functions and buckets."""

import contextlib

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
