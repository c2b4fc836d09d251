"""Tensors stored column by column (transposed matrices) against the CPU checker, by bytes."""

import pytest
import torch

from test_gpu_parity import NT, q, same_bytes  # noqa: F401 (q is a fixture)

pytestmark = pytest.mark.gpu


def transposed(m, n, gap, off, dtype, g, device="cpu"):
    """An [m, n] view with columns of m elements, `gap` elements apart, `off` elements into its
    storage, and the storage, which is 9 outside the view."""
    base = torch.full((off + n * (m + gap) + 3,), 9.0, dtype=dtype)
    view = torch.as_strided(base, (m, n), (1, m + gap), off)
    x = torch.randn(m, n, generator=g)
    x[m // 2] *= 1e-30   # a scale that takes the plain divide
    x[m // 3] = 0.0
    view.copy_((x * 0.1).to(dtype))
    return view, base


# rows on both sides of a lane's 4 or 8, a block's 8 or 16 and a tile's 64; columns on both sides of
# a tile's 256, a step's 1024 and of what stays in the registers (4 and 12 steps)
SHAPES = [(8, 17), (9, 18), (15, 256), (16, 257), (17, 255), (63, 300), (64, 1024), (65, 1025), (130, 1023),
          (24, 2049), (40, 4096), (33, 4099), (21, 12288), (19, 12289), (37, 14001), (200, 64), (1000, 33)]


@pytest.mark.parametrize("ws", [1, 3, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("long_list", [False, True])
def test_transposed_matrices(q, oracle, dtype, ws, long_list):  # noqa: F811
    g = torch.Generator().manual_seed(ws)
    shapes = SHAPES if long_list else SHAPES[ws::3]
    views, bases = zip(*[transposed(m, n, i % 3, i % 5, dtype, g) for i, (m, n) in enumerate(shapes)])
    views, bases = list(views), list(bases)
    rows = torch.randn(50, 300, generator=g).to(dtype)  # and one that is stored row by row
    tensors = views + [rows]
    packed = oracle.fused_quantize_into_fp8([t.clone() for t in tensors], ws, nthreads=NT)
    gpu_bases = [b.cuda() for b in bases]
    gpu_views = [torch.as_strided(b, v.shape, v.stride(), v.storage_offset()) for b, v in zip(gpu_bases, views)]
    gpu = gpu_views + [rows.cuda()]
    same_bytes(q.fused_quantize_into_fp8(list(gpu), ws), packed, "quantize")
    for b in gpu_bases + bases:
        b.fill_(9.0)
    q.fused_dequantize_from_fp8(list(gpu), packed.cuda(), ws)
    oracle.fused_dequantize_from_fp8(list(tensors), packed, ws, nthreads=NT)
    for i, (b, c) in enumerate(zip(gpu_bases, bases)):
        same_bytes(b, c, f"dequantize {shapes[i]} with its guard elements")
    q.fused_dequantize_from_fp8(list(gpu), packed.cuda(), ws, divide_by=3)
    for v, c, s in zip(gpu_views, views, shapes):  # (torch drops the sign of some fp16 zeros: compared as numbers)
        assert torch.equal(v, c.cuda() / 3), f"dequantize and divide {s}"


def test_reduce_static_takes_2800_transposed_tensors():
    """The index of quantize's second launch, which reduce does not read, is not part of what has to
    fit the library's fixed array: a list whose whole table does not."""
    import ctypes

    from torchft_amd import _lib
    L = _lib.load()
    T, m, n, ws, rank = 2800, 1000, 400, 2, 1
    shapes = (ctypes.c_int64 * (2 * T))(*([m, n] * T))
    strides = (ctypes.c_int64 * (2 * T))(*([1, m] * T))
    h = ctypes.c_void_p()
    assert L.tftq_plan_create(2, T, shapes, strides, ws, ctypes.byref(h)) == 0
    size, nbytes = L.tftq_plan_output_size(h), L.tftq_plan_table_bytes(h)
    assert nbytes > 512 * 1024
    x = (torch.randn(n, m, generator=torch.Generator().manual_seed(1)) * 0.1).to(torch.bfloat16).cuda()
    host = (ctypes.c_uint8 * nbytes).from_address(L.tftq_plan_table_host(h))
    table = torch.frombuffer(host, dtype=torch.uint8).cuda()
    pointers = torch.full((T,), x.data_ptr(), dtype=torch.int64, device="cuda")  # one matrix 2800 times
    a = torch.empty(size, dtype=torch.uint8, device="cuda")
    stream, dev = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), torch.cuda.current_device()
    assert L.tftq_quantize(h, None, table.data_ptr(), pointers.data_ptr(), a.data_ptr(), size, dev, stream) == 0
    b = a.clone()
    assert L.tftq_reduce(h, table.data_ptr(), a.data_ptr(), size, rank, 1, dev, stream) == 0
    assert L.tftq_reduce_static(h, b.data_ptr(), size, rank, 1, dev, stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    L.tftq_plan_destroy(h)
