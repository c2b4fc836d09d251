"""Lists of one tensor: their kernels find their work without the tables of longer lists."""

import os
import subprocess

import pytest
import torch
from torch.distributed import ReduceOp

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_every_block_is_visited_once(tmp_path):
    exe = str(tmp_path / "one_piece")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-o", exe,
                           os.path.join(HERE, "one_piece.cpp"), os.path.join(ROOT, "torchft_amd", "csrc", "tftq_plan.cpp")])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape, layout", [
    ((1,), "rows"), ((5003,), "rows"), ((5003,), "every other"), ((7, 2), "rows"), ((1030, 19), "rows"), ((65, 300), "rows"),
    ((33, 1000), "rows"), ((257, 4096), "rows"), ((40, 9001), "rows"), ((9, 20001), "rows"), ((5, 70003), "rows"),
    ((65, 300), "slice"), ((300, 65), "columns"), ((2048, 5000), "columns"), ((33, 130), "every other"),
])
def test_same_bytes_as_among_others(shape, layout, dtype):
    """One tensor alone against the same tensor in front of another one, all three stages."""
    import torchft_amd

    def tensor(generator):
        wide = [2 * s for s in shape]
        if layout == "rows":
            t = torch.empty(shape, dtype=dtype, device="cuda")
        elif layout == "columns":
            t = torch.empty(shape[::-1], dtype=dtype, device="cuda").t()
        elif layout == "slice":
            t = torch.empty((shape[0], wide[1]), dtype=dtype, device="cuda")[:, 1:1 + shape[1]]
        else:
            t = torch.empty(wide, dtype=dtype, device="cuda")[tuple(slice(None, None, 2) for _ in shape)]
        return t.copy_(torch.randn(shape, generator=generator, device="cuda") * 0.02)

    generator = torch.Generator("cuda").manual_seed(1)
    other = torch.ones(1, 4, dtype=dtype, device="cuda")
    for ws, op in ((1, ReduceOp.SUM), (2, ReduceOp.AVG), (3, ReduceOp.AVG), (8, ReduceOp.SUM), (70, ReduceOp.AVG), (1030, ReduceOp.AVG)):
        t = tensor(generator)
        alone, among = [t], [t, other]
        a = torchft_amd.fused_quantize_into_fp8(alone, ws)
        b = torchft_amd.fused_quantize_into_fp8(among, ws)
        part = a.numel() // ws  # a slot of the longer list starts with the tensor's rows

        def same(a, b):
            return torch.equal(a.view(ws, -1), b.view(ws, -1)[:, :part])

        assert same(a, b)
        a.view(ws, -1)[0].copy_(a.view(ws, -1)[-1].clone())
        b.view(ws, -1)[0].copy_(b.view(ws, -1)[-1].clone())
        rank = ws // 2
        torchft_amd.fused_reduce_fp8(alone, a, ws, rank, op)
        torchft_amd.fused_reduce_fp8(among, b, ws, rank, op)
        assert same(a, b)
        for divide_by in (None, 3):
            torchft_amd.fused_dequantize_from_fp8(alone, a, ws, divide_by=divide_by)
            got = t.clone(memory_format=torch.contiguous_format)
            t.zero_()
            torchft_amd.fused_dequantize_from_fp8(among, b, ws, divide_by=divide_by)
            now = t.clone(memory_format=torch.contiguous_format)
            assert torch.equal(got.view(-1).view(torch.uint8), now.view(-1).view(torch.uint8))
