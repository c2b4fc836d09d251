"""Reduce of rows of 129 to 1024 dwords of codes in groups of 5 to 64 peers, tensors of a few rows
and of rows enough for the smaller teams, against the CPU checker, by bytes."""

import pytest
import torch
from torch.distributed import ReduceOp

from test_gpu_parity import NT, q, same_bytes  # noqa: F401 (q is a fixture)

pytestmark = pytest.mark.gpu

# dwords of codes on both sides of the teams' lines
DWORDS = [33, 64, 65, 128, 129, 192, 193, 256, 257, 384, 385, 512, 513, 768, 769, 1024, 1025]


def check(q, oracle, shapes, ws, op, plain_divide=False):  # noqa: F811
    g = torch.Generator().manual_seed(ws)
    tensors = [torch.randn(s, generator=g) * 0.1 for s in shapes]
    for i, t in enumerate(tensors):
        t[len(t) // 3] = -0.0
        if plain_divide and i % 2:
            t[len(t) // 2] *= 1e-30  # a scale outside the range of the fast division
    gpu = [t.to(torch.bfloat16).cuda() for t in tensors]
    received = q.fused_quantize_into_fp8(list(gpu), ws)  # what the peers sent: slots that differ
    for rank in (0, ws - 1):
        packed, host = received.clone(), received.cpu()
        q.fused_reduce_fp8(gpu, packed, ws, rank, op)
        oracle.fused_reduce_fp8([torch.empty(s, dtype=torch.bfloat16) for s in shapes], host, ws, rank, op, nthreads=NT)
        same_bytes(packed, host, f"rank {rank}")


@pytest.mark.parametrize("plain_divide", [False, True])
@pytest.mark.parametrize("long_list", [False, True])
@pytest.mark.parametrize("ws,op", [(5, ReduceOp.AVG), (8, ReduceOp.SUM), (9, ReduceOp.AVG), (12, ReduceOp.SUM), (13, ReduceOp.AVG),
                                   (16, ReduceOp.AVG), (17, ReduceOp.AVG), (24, ReduceOp.SUM), (25, ReduceOp.AVG),
                                   (32, ReduceOp.SUM), (33, ReduceOp.AVG), (49, ReduceOp.SUM), (64, ReduceOp.AVG)])
def test_a_few_rows(q, oracle, ws, op, long_list, plain_divide):  # noqa: F811
    shapes = [(ws * (i % 5) + 1 + i % ws, 4 * d - i % 4) for i, d in enumerate(DWORDS)]
    for some in ([shapes] if long_list else [shapes[:9], shapes[9:], shapes[4:5], shapes[13:14]]):
        check(q, oracle, some, ws, op, plain_divide)


@pytest.mark.parametrize("ws,dwords,per_slot", [(5, 175, 4096), (4, 175, 2048), (3, 175, 511), (9, 190, 4095), (9, 375, 512), (5, 500, 511),
                                                (13, 500, 767), (13, 375, 768), (9, 640, 1279), (9, 640, 1280), (6, 750, 1024), (5, 640, 512)])
def test_rows_enough_for_smaller_teams(q, oracle, ws, dwords, per_slot):  # noqa: F811
    check(q, oracle, [(per_slot * ws - 1, 4 * dwords - 1)], ws, ReduceOp.AVG)
