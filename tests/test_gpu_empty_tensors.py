"""Empty tensors in long lists, in front of rows that need a whole workgroup in reduce, against the
CPU checker, by bytes."""

import pytest
import torch
from torch.distributed import ReduceOp

from test_gpu_parity import full_check, q  # noqa: F401 (q is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ws,op", [(2, ReduceOp.SUM), (8, ReduceOp.AVG), (17, ReduceOp.SUM), (33, ReduceOp.AVG), (70, ReduceOp.SUM)])
@pytest.mark.parametrize("n", [0, 1, 3, 5, 12, 16, 24, 60, 100, 250, 500])  # a row length per kind of reduce
def test_empty_tensors_in_long_lists(q, oracle, n, ws, op):  # noqa: F811
    shapes = [(0, n), (5, n + 1), (5, 2100), (0, 3000), (2 * ws + 1, 5000), (0, n)] + [(5, 4)] * 14
    g = torch.Generator().manual_seed(n)
    base = [[(torch.randn(s, generator=g) * (1 + p)).to(torch.bfloat16) for s in shapes] for p in range(min(ws, 3))]
    full_check(q, oracle, [base[p % len(base)] for p in range(ws)], ws, op, sorted({0, ws - 1}))
