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


def kinds(shapes, ws, dtype):
    """The lane mappings of quantize and dequantize (kind[0] and kind[2] of the 64-byte descriptors) that
    a long list of transposed tensors gets."""
    import ctypes

    from torchft_amd import _lib
    L = _lib.load()
    T = len(shapes)
    h = ctypes.c_void_p()
    assert L.tftq_plan_create({torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype], T,
                              (ctypes.c_int64 * (2 * T))(*[d for s in shapes for d in s]),
                              (ctypes.c_int64 * (2 * T))(*[d for s in shapes for d in (1, s[0])]), ws, ctypes.byref(h)) == 0
    table = (ctypes.c_uint8 * (64 * T)).from_address(L.tftq_plan_table_host(h))
    got = [(table[64 * i + 60], table[64 * i + 62]) for i in range(T)]
    L.tftq_plan_destroy(h)
    return got


# rows on both sides of the 4 or 8 of a lane, the 8 or 16 of a block and the 64 of a tile, per slot;
# columns on both sides of a tile's 256, a step's 1024 and of what stays in the registers
EDGES = [(8, 1024), (9, 1025), (15, 1023), (16, 2049), (17, 2048), (31, 1536), (33, 4099), (63, 767), (64, 900), (65, 1281),
         (129, 511), (12, 12289), (24, 12288), (40, 13001), (128, 513), (191, 257), (300, 256)]


@pytest.mark.parametrize("ws", [1, 2, 5, 16])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("count", [1, 16, 17])
def test_nothing_but_transposed_matrices(q, oracle, dtype, ws, count):  # noqa: F811
    g = torch.Generator().manual_seed(ws)
    shapes = [(m * ws - i % 2 * (ws > 1) if m * n < 1 << 17 else m, n) for i, (m, n) in enumerate(EDGES)]
    assert set(kinds(shapes, ws, dtype)) == {(17, 18)}
    for at in (range(len(shapes)) if count == 1 else [0]):
        part = (shapes[at:] + shapes)[:count]
        views, bases = zip(*[transposed(m, n, i % 3, (at + i) % 5, dtype, g) for i, (m, n) in enumerate(part)])
        packed = oracle.fused_quantize_into_fp8([v.clone() for v in views], ws, nthreads=NT)
        gpu_bases = [b.cuda() for b in bases]
        gpu = [torch.as_strided(b, v.shape, v.stride(), v.storage_offset()) for b, v in zip(gpu_bases, views)]
        same_bytes(q.fused_quantize_into_fp8(list(gpu), ws), packed, f"quantize {part}")
        for b in [*gpu_bases, *bases]:
            b.fill_(9.0)
        q.fused_dequantize_from_fp8(list(gpu), packed.cuda(), ws)
        oracle.fused_dequantize_from_fp8(list(views), packed, ws, nthreads=NT)
        for b, c, s in zip(gpu_bases, bases, part):
            same_bytes(b, c, f"dequantize {s} with its guard elements")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n", [(64, 64), (130, 36), (9, 128), (100, 127), (33, 65), (70, 100)])
def test_one_narrow_transposed_matrix(q, oracle, dtype, m, n):  # noqa: F811
    """Few columns: the blocks where the machine takes the whole list at once."""
    g = torch.Generator().manual_seed(n)
    for ws in (1, 3, 8):
        v, b = transposed(m, n, 1, 3, dtype, g)
        packed = oracle.fused_quantize_into_fp8([v.clone()], ws)
        d = b.cuda()
        gpu = torch.as_strided(d, v.shape, v.stride(), v.storage_offset())
        same_bytes(q.fused_quantize_into_fp8([gpu], ws), packed, "quantize")
        d.fill_(9.0)
        b.fill_(9.0)
        q.fused_dequantize_from_fp8([gpu], packed.cuda(), ws)
        oracle.fused_dequantize_from_fp8([v], packed, ws)
        same_bytes(d, b, "dequantize")
