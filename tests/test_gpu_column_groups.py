"""Transposed matrices in quantize's blocks of 2 to 32 groups of rows against the CPU checker, by bytes."""

import pytest
import torch

from test_gpu_columns import transposed
from test_gpu_parity import NT, q, same_bytes  # noqa: F401 (q is a fixture)

pytestmark = pytest.mark.gpu

# (rows per slot, columns): rows on both sides of the 4 or 8 of a lane and of the blocks of 8 to 256, columns
# on both sides of one, two and four steps (of 64, 128, 256, 512 and 1024 columns) and of twelve of 512
EDGES = [(513, 17), (256, 64), (255, 65), (257, 129), (300, 33), (129, 256), (128, 257), (127, 511), (65, 1025),
         (130, 600), (33, 2048), (31, 2049), (65, 3000), (200, 6144), (50, 6145), (300, 40), (7, 4097)]


@pytest.mark.parametrize("ws", [1, 3, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("together", [False, True])
def test_groups_of_rows(q, oracle, dtype, ws, together):  # noqa: F811
    """Each alone, where a block is chosen for its latency too, and all in one list, where it is chosen for
    the least work; the last slot is one row short, and offsets and gaps leave no column aligned."""
    g = torch.Generator().manual_seed(ws)
    views = [transposed(max(8, m * ws - (ws > 1)), n, i % 3, i % 5, dtype, g)[0] for i, (m, n) in enumerate(EDGES)]
    for part in [views] if together else [[v] for v in views]:
        packed = oracle.fused_quantize_into_fp8([v.clone() for v in part], ws, nthreads=NT)
        gpu = [torch.empty(v.stride(1) * v.shape[1] + 8, dtype=dtype, device="cuda")[v.storage_offset():]
               .as_strided(v.shape, v.stride(), v.storage_offset()) for v in part]
        for a, b in zip(gpu, part):
            a.copy_(b)
        same_bytes(q.fused_quantize_into_fp8(gpu, ws), packed, f"{[tuple(v.shape) for v in part]}")


# slots and lists of 2 groups: launches of at most and of more than 48 blocks of rows of 5 to 8 steps and 192 of
# rows of 1 to 4, alone and in lists, each number of steps at both ends and rows of more than 12
FEW = [(1, [(768, 7001)]), (1, [(784, 7001)]), (1, [(3072, 2049)]), (1, [(3088, 2049)]), (3, [(130, 1024)]),
       (3, [(133, 1025), (65, 2049), (40, 2048)]), (2, [(100, 4096), (31, 17), (64, 5000)]), (8, [(384, 8192)]),
       (8, [(383, 8192), (70, 4097)]), (1, [(784, 8192), (16, 14000)]), (2, [(700, 8193), (33, 900)])]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ws, shapes", FEW)
def test_few_blocks(q, oracle, dtype, ws, shapes):  # noqa: F811
    """Rows straight from the registers: every element is in the maximum whatever the number of steps (each
    row's largest is in its last column)."""
    g = torch.Generator().manual_seed(len(shapes))
    views = [transposed(m, n, i % 3, i % 5, dtype, g)[0] for i, (m, n) in enumerate(shapes)]
    for v in views:
        v[:, -1] = 3.0 + torch.arange(v.shape[0]).to(dtype) / 1024
    packed = oracle.fused_quantize_into_fp8([v.clone() for v in views], ws, nthreads=NT)
    gpu = [torch.empty(v.stride(1) * v.shape[1] + 8, dtype=dtype, device="cuda")[v.storage_offset():]
           .as_strided(v.shape, v.stride(), v.storage_offset()) for v in views]
    for a, b in zip(gpu, views):
        a.copy_(b)
    same_bytes(q.fused_quantize_into_fp8(gpu, ws), packed, f"{shapes}")
