"""Reduce of short rows in groups of more peers than a team of lanes or its registers hold at
once, and of one-column tensors of few rows, against the CPU checker, by bytes."""

import pytest
import torch
from torch.distributed import ReduceOp

from test_gpu_parity import full_check, q  # noqa: F401 (q is a fixture)

pytestmark = pytest.mark.gpu

# columns on both sides of 1, 2, 3, 4, 8, 12, 16, 32, 64 and 128 dwords of codes
COLUMNS = [0, 1, 2, 4, 5, 8, 9, 12, 13, 16, 17, 31, 32, 33, 44, 45, 48, 49, 64, 65, 127, 128, 129, 256, 257, 511, 512]


@pytest.mark.parametrize("plain_divide", [False, True])
@pytest.mark.parametrize("long_list", [False, True])
@pytest.mark.parametrize("ws,op", [(1, ReduceOp.SUM), (2, ReduceOp.AVG), (7, ReduceOp.AVG), (8, ReduceOp.SUM), (9, ReduceOp.AVG),
                                   (16, ReduceOp.AVG), (17, ReduceOp.SUM), (24, ReduceOp.AVG), (25, ReduceOp.SUM),
                                   (33, ReduceOp.AVG), (64, ReduceOp.AVG), (65, ReduceOp.SUM), (70, ReduceOp.AVG)])
def test_short_rows_in_large_groups(q, oracle, ws, op, long_list, plain_divide):  # noqa: F811
    g = torch.Generator().manual_seed(ws)
    columns = COLUMNS if long_list else COLUMNS[ws % 2::2]
    shapes = [((3 * i) % (4 * ws) + 1, n) for i, n in enumerate(columns)]
    base = []
    for p in range(min(ws, 3)):
        ts = [torch.randn(s, generator=g) * (1 + p) for s in shapes]
        for i, t in enumerate(ts):
            t[len(t) // 3] = -0.0
            if plain_divide and p == 1 and i % 2:
                t[len(t) // 2] *= 1e-30  # a scale outside the range of the fast division
        base.append([t.to(torch.bfloat16) for t in ts])
    full_check(q, oracle, [base[p % len(base)] for p in range(ws)], ws, op, sorted({0, ws // 2, ws - 1}))


@pytest.mark.parametrize("ws,op", [(1, ReduceOp.SUM), (2, ReduceOp.SUM), (3, ReduceOp.AVG), (4, ReduceOp.AVG),
                                   (5, ReduceOp.SUM), (16, ReduceOp.AVG), (17, ReduceOp.SUM), (70, ReduceOp.AVG)])
@pytest.mark.parametrize("long_list", [False, True])
def test_one_column_of_few_and_many_rows(q, oracle, ws, op, long_list):  # noqa: F811
    # rows per slot on both sides of a wavefront, a workgroup and four rows per lane
    per_slot = [1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 1280, 1281]
    sizes = [n * ws - i % 2 * (ws > 1) for i, n in enumerate(per_slot)] * (2 if long_list else 1)
    g = torch.Generator().manual_seed(ws)
    base = []
    for p in range(min(ws, 3)):
        ts = [torch.randn(n, generator=g) * 10.0 ** torch.randint(-30, 30, (n,), generator=g).float() for n in sizes]
        for t in ts:
            t[::5] = 0.0
        base.append(ts)
    full_check(q, oracle, [base[p % len(base)] for p in range(ws)], ws, op, sorted({0, ws - 1}))


@pytest.mark.parametrize("plain_divide", [False, True])
@pytest.mark.parametrize("long_list", [False, True])
@pytest.mark.parametrize("ws,op", [(1, ReduceOp.SUM), (2, ReduceOp.AVG), (3, ReduceOp.AVG), (4, ReduceOp.SUM)])
def test_rows_side_by_side_in_small_groups(q, oracle, ws, op, long_list, plain_divide):  # noqa: F811
    # rows per slot on both sides of 256 workgroups of teams of 1, 2, 4, 8, 16 and 32 lanes, and
    # remainders of a wavefront's rows
    shapes = [(65535 * ws, 13), (65537 * ws, 14), (65536 * ws, 16), (32771 * ws, 19), (16383 * ws, 48), (16384 * ws, 46),
              (16389 * ws, 60), (8193 * ws, 65), (8195 * ws, 128), (4101 * ws - ws // 2, 130), (2048 * ws, 511), (2055 * ws, 257)]
    shapes = shapes + [(3, 40)] * 8 if long_list else shapes[ws % 2::2]
    g = torch.Generator().manual_seed(ws)
    peers = []
    for p in range(ws):
        ts = [torch.randn(s, generator=g) * (1 + p) for s in shapes]
        for t in ts:
            t[len(t) // 3] = -0.0
            if plain_divide:
                t[len(t) // 2] *= 1e-30
        peers.append([t.to(torch.bfloat16) for t in ts])
    full_check(q, oracle, peers, ws, op, sorted({0, ws - 1}))


# (columns, rows per slot from which rows go side by side in groups of 1 and of 2: tftq_reduce_rows_side)
SIDE = [(17, 262144, 1048576), (32, 262144, None), (46, 131072, 131072), (60, 131072, 1048576), (65, 32768, 49152),
        (128, 32768, 49152), (130, 16384, 24576), (257, 8192, 12288), (512, 8192, 12288)]


@pytest.mark.parametrize("plain_divide", [False, True])
@pytest.mark.parametrize("ws,op", [(1, ReduceOp.SUM), (2, ReduceOp.AVG)])
@pytest.mark.parametrize("n,one,two", SIDE)
def test_rows_side_by_side_where_workgroups_are_left(q, oracle, n, one, two, ws, op, plain_divide):  # noqa: F811
    least = (one, two)[ws - 1] or 300000
    g = torch.Generator().manual_seed(n)
    shapes = [(least * ws, n), ((least - 1) * ws, n), ((least + 3) * ws - ws // 2, n)]
    for shape in shapes if n < 40 or least < 1 << 20 else shapes[2:]:
        base = torch.randn(1000, n, generator=g)
        base[333] = -0.0
        if plain_divide:
            base[500] *= 1e-30
        peers = [[(base * (1 + p)).to(torch.bfloat16).repeat(-(-shape[0] // 1000), 1)[:shape[0]].contiguous()] for p in range(ws)]
        full_check(q, oracle, peers, ws, op, [ws - 1])


@pytest.mark.parametrize("plain_divide", [False, True])
@pytest.mark.parametrize("long_list", [False, True])
@pytest.mark.parametrize("ws,op", [(9, ReduceOp.SUM), (10, ReduceOp.AVG), (11, ReduceOp.SUM), (12, ReduceOp.AVG), (12, ReduceOp.SUM),
                                   (13, ReduceOp.AVG), (15, ReduceOp.SUM)])
def test_short_rows_in_groups_of_9_to_15(q, oracle, ws, op, long_list, plain_divide):  # noqa: F811
    test_short_rows_in_large_groups(q, oracle, ws, op, long_list, plain_divide)
