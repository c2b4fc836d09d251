"""The work that users of this package have it do, as measurable cases.

One case is one whole quantized all-reduce (or reduce-scatter) of a list of tensors as one rank
sees it: quantize the tensors, reduce the slots that the peers have sent, dequantize what all
ranks have reduced.  ``api`` is the public entry point it goes through:

    functions       the three functions of ``torchft_amd.quantization`` called one after the other,
                    with the peers' buffers at hand (the exchange is not part of the pass)
    prepared        the same through a ``PreparedBucket`` that the program keeps
    managed         ``torchft_amd.allreduce.allreduce`` of one tensor over a process group
    diloco          ``torchft_amd.allreduce.BucketizedAllreduce`` over a process group
    reduce_scatter  ``torchft_amd.reduce_scatter_quantized`` over a process group

The process group of the last three is one rank of a group whose other ranks' bytes lie on the
GPU already: an exchange is one copy of the buffer.

Other keys of a case: ``dtype``; ``ws``, the group size; ``op``, ``sum`` or ``avg``; ``shapes``, a
list as text, ``2*16x4096, 512`` for two matrices and a vector; ``ragged``, instead of ``shapes``:
that many tensors of 1 to 4096 elements and of every row length; ``layout``: ``rows``
(contiguous), ``columns`` (every matrix is the transpose of a contiguous one) or ``slices``
(every matrix is a range of the columns of a wider one).
"""

from __future__ import annotations

import math
import random

import torch
from torch.distributed import ReduceOp

import torchft_amd
from torchft_amd.allreduce import BucketizedAllreduce, allreduce

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_OPS = {"sum": ReduceOp.SUM, "avg": ReduceOp.AVG}
_ALIGN = 256   # bytes: every tensor starts where an allocation of its own could start
_BLOCK = 512   # elements that share one standard deviation
# No drawn case has more elements: a quarter of the largest listed one.
_MOST_DRAWN = 1 << 28


def _case(name, api, dtype, ws, op, shapes="", ragged=0, layout="rows"):
    return {"name": name, "api": api, "dtype": dtype, "ws": ws, "op": op, "shapes": shapes,
            "ragged": ragged, "layout": layout}


def listed():
    return [
        # One norm weight: the smallest call of a per-parameter all-reduce, all of it latency.
        _case("norm weight", "functions", "bfloat16", 8, "avg", "4096"),
        # A layer of a small model with its bias between two replicas (benchmark configuration 1).
        _case("small layer", "functions", "float32", 2, "sum", "256x512, 1024"),
        # One square weight gradient (benchmark configuration 2): one round of workgroups.
        _case("one matrix", "functions", "bfloat16", 8, "avg", "4096x4096"),
        # The gradients of one decoder layer of an 8B model, reduced every step (configuration 3).
        _case("layer bucket", "prepared", "bfloat16", 8, "avg",
              "4096x4096, 2*1024x4096, 4096x4096, 2*14336x4096, 4096x14336, 2*4096"),
        # The pseudo-gradient of a 1.1B model, DiLoCo's outer step over 4 replicas (configuration 4).
        _case("pseudo-gradient", "prepared", "float32", 4, "sum",
              "32000x2048, 44*2048x2048, 44*256x2048, 44*5632x2048, 22*2048x5632, 45*2048, 32000x2048"),
        # Ten thousand small tensors of every shape (configuration 5), 16 replicas.
        _case("ragged list", "functions", "bfloat16", 16, "avg", ragged=10000),
        # One fragment of the 1.1B model through DiLoCo's flat buffer: rows of one column.
        _case("flat bucket", "diloco", "float32", 2, "avg",
              "2*2048x2048, 2*256x2048, 2*5632x2048, 2048x5632, 2*2048"),
        # Rows that are no whole number of vectors, in half precision, three replicas.
        _case("odd rows", "functions", "float16", 3, "avg", "20001x1001, 5003x257, 3001x5003, 1001"),
        # Gradients that come out transposed (weights kept column by column).
        _case("transposed", "functions", "bfloat16", 8, "avg", "4096x14336, 4096x4096", layout="columns"),
        # Low-rank adapters: very short and long rows in one list.
        _case("adapters", "prepared", "bfloat16", 8, "avg", "64*16x4096, 64*4096x16, 64*64x4096, 64*14336x64"),
        # One layer of a 70B-class model: its widest rows do not fit a workgroup's registers.
        _case("wide layer", "prepared", "bfloat16", 16, "sum",
              "8192x8192, 2*1024x8192, 8192x8192, 2*28672x8192, 8192x28672, 2*8192"),
        # A vocabulary table that every rank keeps a share of.
        _case("sharded table", "reduce_scatter", "float32", 4, "sum", "32000x2048"),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5))))))


def draw(rng):
    family = rng.choice(["vector", "matrix", "matrix", "few", "few", "adapters", "ragged", "strided", "group"])
    case = _case("", "functions", rng.choice(["bfloat16", "bfloat16", "float32", "float16"]),
                 rng.choice([1, 2, 2, 3, 4, 5, 6, 7, 8, 8, 8, 12, 16, 16, 24, 32, 64]), rng.choice(["sum", "avg"]))
    del case["name"]
    case["api"] = rng.choice(["functions", "prepared"])
    if family == "vector":
        case["shapes"] = str(_spread(rng, 64, 1 << 26))
    elif family == "matrix":
        cols = _spread(rng, 2, 57344)
        rows = _spread(rng, 1, max(1, _MOST_DRAWN // cols))
        case["shapes"] = f"{rows}x{cols}"
    elif family == "few":
        width = _spread(rng, 64, 16384)
        items, left = [], _MOST_DRAWN
        for _ in range(rng.randint(2, 12)):
            cols = rng.choice([width, width, 4 * width, max(1, width // 3), 0])
            if cols == 0:
                items.append(str(width))
                continue
            rows = _spread(rng, 8, 16384)
            if rows * cols <= left:
                left -= rows * cols
                items.append(f"{rows}x{cols}")
        case["shapes"] = ", ".join(items) or str(width)
    elif family == "adapters":
        rank, width, count = rng.choice([4, 8, 16, 32, 64, 128]), _spread(rng, 512, 8192), rng.randint(4, 128)
        case["shapes"] = f"{count}*{rank}x{width}, {count}*{width}x{rank}"
    elif family == "ragged":
        case["ragged"] = _spread(rng, 17, 20000)
        case["ws"] = min(case["ws"], 16)
    elif family == "strided":
        cols = _spread(rng, 8, 16384)
        rows = _spread(rng, 64, max(64, (_MOST_DRAWN >> 2) // cols))
        case["shapes"] = f"{rows}x{cols}"
        case["layout"] = rng.choice(["columns", "columns", "slices"])
    else:
        case["api"] = rng.choice(["managed", "diloco", "reduce_scatter"])
        case["ws"] = min(case["ws"], 8)
        if case["api"] != "reduce_scatter":
            case["op"] = "avg"  # in place, pass after pass: sums would grow without end
        if case["api"] == "diloco":
            case["ws"] = max(2, min(case["ws"], 4))
            width = _spread(rng, 256, 4096)
            case["shapes"] = f"{rng.randint(1, 4)}*{width}x{width}, {_spread(rng, 64, 4096)}x{width}, 2*{width}"
        else:
            cols = _spread(rng, 64, 16384)
            case["shapes"] = f"{_spread(rng, 64, 1 << 14)}x{cols}"
    return case


def _shapes(case):
    """The list's shapes, (rows, columns); a vector has one number."""
    if case["ragged"]:
        rng, out = random.Random(case["ragged"]), []
        for _ in range(case["ragged"]):
            n, kind = rng.randint(1, 4096), rng.randrange(8)
            if kind == 0:
                out.append((n,))
                continue
            cols = rng.randint(1, 3) if kind == 1 else n if kind == 2 else rng.randint(1, max(1, min(n, 600)))
            out.append((max(1, n // cols), cols))
        return out
    out = []
    for item in case["shapes"].split(","):
        times, _, shape = item.strip().rpartition("*")
        out += [tuple(int(x) for x in shape.split("x"))] * int(times or 1)
    return out


def _tensors(case, shapes):
    """The tensors, uninitialised, and the one buffer that they are all views of."""
    dtype = _DTYPES[case["dtype"]]
    unit = _ALIGN // dtype.itemsize
    extents, total = [], 0
    for s in shapes:
        n = math.prod(s)
        if len(s) == 2 and case["layout"] == "slices":
            n = s[0] * (s[1] + s[1] // 2)
        extents.append((total, n))
        total += -(-n // unit) * unit
    flat = torch.empty(-(-total // _BLOCK) * _BLOCK, dtype=dtype, device="cuda")
    tensors = []
    for s, (at, n) in zip(shapes, extents):
        part = flat[at:at + n]
        if len(s) == 1:
            tensors.append(part)
        elif case["layout"] == "columns":
            tensors.append(part.view(s[1], s[0]).t())
        elif case["layout"] == "slices":
            tensors.append(part.view(s[0], -1)[:, :s[1]])
        else:
            tensors.append(part.view(s))
    return tensors, flat


def _fill(flat, generator):
    """Gradients: normal, with a standard deviation that differs by up to three decades from one
    place to the next, and here and there nothing at all (rows of a table that no token used)."""
    flat.normal_(generator=generator)
    blocks = flat.view(-1, _BLOCK)
    draw = torch.rand(blocks.shape[0], 1, device=flat.device, generator=generator)
    std = torch.where(draw < 0.01, 0.0, 10.0 ** (3.0 * draw - 4.0))
    blocks.mul_(std.to(flat.dtype))


class _Done:
    """A collective that is complete in stream order."""

    def wait(self, timeout=None):
        return True

    def get_future(self):
        future = torch.futures.Future()
        future.set_result(None)
        return future


class _Group:
    """Rank 0 of a group: the other ranks' bytes are those of `received` and `gathered`."""

    def __init__(self, received, gathered):
        self.received, self.gathered = received, gathered

    def rank(self):
        return 0

    def size(self):
        return self.received.shape[0]

    def alltoall_base(self, output, input, output_splits, input_splits, opts=None):
        output[1:].copy_(self.received[1:])
        output[0].copy_(input[0])
        return _Done()

    def allgather_into_tensor_coalesced(self, outputs, inputs, opts=None):
        outputs[0][1:].copy_(self.gathered[1:])
        outputs[0][:1].copy_(inputs[0])
        return _Done()


def prepare(case, seed):
    generator = torch.Generator("cuda").manual_seed(seed)
    api, ws = case["api"], case["ws"]
    rank = 0 if api in ("managed", "diloco", "reduce_scatter") else ws // 2
    tensors, flat = _tensors(case, _shapes(case))
    # what goes over the wire: DiLoCo's flat buffer instead of the tensors
    wire = [torch.empty(sum(t.numel() for t in tensors), dtype=flat.dtype, device="cuda")] if api == "diloco" else tensors
    received = None
    for peer in range(ws):  # slot `rank` of every peer's buffer
        _fill(flat, generator)
        if api == "diloco":
            torch.cat([t.reshape(-1) for t in tensors], out=wire[0])
        packed = torchft_amd.fused_quantize_into_fp8(list(wire), ws)
        if received is None:
            received = torch.empty_like(packed)
        received.view(ws, -1)[peer].copy_(packed.view(ws, -1)[rank])
    _fill(flat, generator)
    state = {"api": api, "ws": ws, "rank": rank, "op": _OPS[case["op"]], "tensors": tensors, "flat": flat,
             "received": received, "gathered": packed}
    if api == "prepared":
        state["bucket"] = torchft_amd.prepare(tensors, ws)
    elif api in ("managed", "diloco", "reduce_scatter"):
        state["group"] = _Group(received.view(ws, -1), packed.view(ws, -1))
    if api == "diloco":
        state["averaging"] = BucketizedAllreduce(tensors, flat.numel() * flat.element_size())
    elif api == "reduce_scatter":
        state["output"] = torchft_amd.allocate_reduce_scatter_output(tensors, ws)[0].zero_()
    return state


def run(state):
    api, tensors, ws = state["api"], state["tensors"], state["ws"]
    if api == "functions":
        packed = torchft_amd.fused_quantize_into_fp8(tensors, ws)
        torchft_amd.fused_reduce_fp8(tensors, state["received"], ws, state["rank"], state["op"])
        torchft_amd.fused_dequantize_from_fp8(tensors, state["gathered"], ws)
        return {"packed": packed, "reduced": state["received"], "tensors": state["flat"]}
    if api == "prepared":
        bucket = state["bucket"]
        packed = bucket.quantize()
        bucket.reduce(state["received"], state["rank"], state["op"])
        bucket.dequantize(state["gathered"])
        return {"packed": packed, "reduced": state["received"], "tensors": state["flat"]}
    if api == "managed":
        allreduce(tensors[0], state["group"], ws, should_quantize=True, reduce_op=state["op"]).wait()
        return state["flat"]
    if api == "diloco":
        for work in state["averaging"].allreduce(state["group"], ws, reduce_op=state["op"]):
            work.wait()
        return state["flat"]
    torchft_amd.reduce_scatter_quantized(state["output"], tensors, state["op"], state["group"],
                                         torch.cuda.current_stream()).wait()
    return state["output"]


def work(case):
    """Quantize reads the tensors and writes the packed buffer; reduce reads the packed buffer and
    writes a slot; dequantize reads the packed buffer (reduce-scatter: a slot) and writes the tensors
    (a share of them)."""
    ws, esz = case["ws"], _DTYPES[case["dtype"]].itemsize
    shapes = _shapes(case)
    if case["api"] == "diloco":
        shapes = [(sum(math.prod(s) for s in shapes),)]
    elements = packed = 0
    for s in shapes:
        m, n = s if len(s) == 2 else (s[0], 1)
        elements += m * n
        packed += -(-m // ws) * ws * (-(-n // 4) * 4 + 4)
    part = ws if case["api"] == "reduce_scatter" else 1
    moved = elements * esz + packed + packed + packed // ws + (packed + elements * esz) // part
    # quantize: maximum and product; reduce: quotient and sum per peer, maximum, product; dequantize: quotient
    return {"bytes": moved, "flops": 2 * elements + 2 * elements + 2 * (elements // ws) + elements // part}


def tolerance(case):
    """The codes and scales are IEEE single precision arithmetic in a fixed order and the tensors
    are their exact quotients: every correct implementation gives the same bytes (measured
    against the oracle on all three types, every row length class and group size: no byte differs)."""
    return "exact"
