"""The kinds for little work (short rows and rows of one column with less work per lane) and the
kinds they take the place of, on both sides of the planner's lines, against the CPU checker, by bytes."""

import pytest
import torch
from torch.distributed import ReduceOp

from test_gpu_parity import NT, full_check, q, same_bytes  # noqa: F401 (q is a fixture)

pytestmark = pytest.mark.gpu


def rows_per_workgroup(n, esz, vecs):
    nvec = -(-n * esz // 16)
    lt = 0
    while lt < (5 if nvec >= 25 else 4) and (1 << lt) < nvec:
        lt += 1
    return (256 >> lt) * (vecs // -(-nvec // (1 << lt)))


@pytest.mark.parametrize("more", [False, True])
@pytest.mark.parametrize("ws", [1, 3, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_short_rows(q, oracle, dtype, ws, more):  # noqa: F811
    """Rows of 1 to 32 vectors, whole or not, in tensors of a workgroup's rows of either kind, one
    more and one less, contiguous and not; `more`: beside a tensor that keeps the machine busy, so
    that only tensors of less than a workgroup get the kind for little work."""
    esz = dtype.itemsize
    g = torch.Generator().manual_seed(ws)
    for nvec in (1, 2, 3, 5, 8, 9, 16, 17, 24, 25, 32):
        n_whole = nvec * 16 // esz
        tensors = []
        for n in (n_whole, n_whole - 1 if nvec > 1 else n_whole, max(16 // esz, n_whole - 16 // esz + 1)):
            for vecs in (2, 8):
                per = rows_per_workgroup(n, esz, vecs)
                for m in (1, per - 1, per + 1):
                    wide = torch.randn(m, n + 3, generator=g).to(dtype)
                    wide[m // 2] *= 1e-30 if dtype != torch.float16 else 0.0
                    tensors.append(wide[:, 1:1 + n] if len(tensors) % 4 == 3 else wide[:, :n].contiguous())
        if more:
            tensors.append(torch.randn(4096, 1024 * 4 // esz, generator=g).to(dtype))
        for some in (tensors[:8] + tensors[18:], tensors):
            gpu = [torch.empty_strided(t.shape, t.stride(), dtype=dtype, device="cuda").copy_(t) for t in some]
            packed = oracle.fused_quantize_into_fp8([t.clone() for t in some], ws, nthreads=NT)
            same_bytes(q.fused_quantize_into_fp8(gpu, ws), packed, f"quantize {nvec} vectors")
            want = [torch.zeros_like(t) for t in some]
            for t in gpu:
                t.zero_()
            oracle.fused_dequantize_from_fp8(want, packed, ws, nthreads=NT)
            q.fused_dequantize_from_fp8(gpu, packed.cuda(), ws)
            for a, b in zip(gpu, want):
                same_bytes(a, b, f"dequantize {tuple(b.shape)}")


@pytest.mark.parametrize("more", [False, True])
@pytest.mark.parametrize("ws,op", [(1, ReduceOp.SUM), (2, ReduceOp.AVG), (3, ReduceOp.AVG), (4, ReduceOp.SUM), (5, ReduceOp.AVG),
                                   (16, ReduceOp.AVG), (17, ReduceOp.SUM), (33, ReduceOp.AVG), (70, ReduceOp.SUM)])
def test_rows_of_one_column(q, oracle, ws, op, more):  # noqa: F811
    """Vectors alone and with matrices; `more`: with rows enough for the other kinds."""
    g = torch.Generator().manual_seed(ws)
    sizes = [1, 255, 511, 513, 1024 * ws - 1, 1024 * ws + 1, 5003]
    if more:
        sizes.append((262144 if ws <= 8 else 524288 // (2 if ws > 32 else 1)) * ws)
    for matrix in ([], [(33, 130)], [(9, 5000)]):
        base = []
        for p in range(min(ws, 3)):
            ts = [torch.randn(n, generator=g) * 10.0 ** (n % 7 - 3) for n in sizes] + [torch.randn(s, generator=g) for s in matrix]
            for t in ts:
                t.view(-1)[::7] = 0.0
            base.append([t.to(torch.bfloat16) for t in ts])
        if more and ws > 8:   # too long a list of peers to check in full: one rank
            ts = [t.cuda() for t in base[0]]
            packed = q.fused_quantize_into_fp8(list(ts), ws)
            host = packed.cpu()
            q.fused_reduce_fp8(ts, packed, ws, ws - 1, op)
            oracle.fused_reduce_fp8(list(base[0]), host, ws, ws - 1, op, nthreads=NT)
            same_bytes(packed, host, "reduce")
        else:
            full_check(q, oracle, [base[p % len(base)] for p in range(ws)], ws, op, sorted({0, ws - 1}))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_strided_vectors(q, oracle, dtype):  # noqa: F811
    for n in (1, 300, 513, 2049, 70001):
        full_check(q, oracle, [[torch.randn(2 * n).to(dtype)[::2], torch.randn(3 * n).to(dtype)[::3]] for _ in range(2)], 2, ReduceOp.AVG)
