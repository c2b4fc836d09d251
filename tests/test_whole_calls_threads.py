"""The whole calls of _pylist beside other threads: what they leave to them, and several at once."""

import os
import subprocess
import sys
import threading

import pytest
import torch
from torch.distributed import ReduceOp

import torchft_amd
from torchft_amd import quantization as q

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# An allocator that notes whether its caller holds the interpreter.
ALLOCATOR = r"""
#include <stddef.h>
#include <sys/types.h>
extern int PyGILState_Check(void);
static int (*hip_malloc)(void **, size_t), (*hip_free)(void *);
int calls, held;
void use(void *m, void *f) { hip_malloc = (int (*)(void **, size_t))m; hip_free = (int (*)(void *))f; }
void *noting_malloc(ssize_t size, int device, void *stream)
{
    void *p = 0;
    calls++;
    held = PyGILState_Check();
    return hip_malloc(&p, size ? size : 1) ? 0 : p;
}
void noting_free(void *p, ssize_t size, int device, void *stream) { hip_free(p); }
"""

PROGRAM = r"""
import ctypes, sys
import torch
from torchft_amd import _lib, quantization as q

lib, noting = _lib.load(), ctypes.CDLL(sys.argv[1])
noting.use(ctypes.cast(lib.hipMalloc, ctypes.c_void_p), ctypes.cast(lib.hipFree, ctypes.c_void_p))
torch.cuda.memory.change_current_allocator(
    torch.cuda.memory.CUDAPluggableAllocator(sys.argv[1], "noting_malloc", "noting_free"))
calls, held = ctypes.c_int.in_dll(noting, "calls"), ctypes.c_int.in_dll(noting, "held")
ts = [torch.randn(64, 512).cuda()]
want = q.fused_quantize_into_fp8(ts, 2)  # the plan becomes known
bucket = q.prepare(ts, 2)
held.value = 1
torch.empty(8, device="cuda")
assert held.value == 0, "torch.empty"

def refuse(*_):
    raise AssertionError("not a whole call")
q._match_short_list = q._check = refuse
for call in (lambda: q.fused_quantize_into_fp8(ts, 2), bucket.quantize):
    held.value, before = -1, calls.value
    got = call()
    assert calls.value == before + 1 and held.value == 0, (calls.value - before, held.value)
    assert torch.equal(got, want)
print("ok")
"""


@pytest.mark.gpu
def test_other_threads_run_during_the_allocation(tmp_path):
    """torch.empty gives up the interpreter before it asks the allocator, which may have to wait for the GPU."""
    if q._pylist is None:
        pytest.skip("torchft_amd._pylist is not built")
    (tmp_path / "noting.c").write_text(ALLOCATOR)
    so = str(tmp_path / "noting.so")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "noting.c")])
    res = subprocess.run([sys.executable, "-c", PROGRAM, so], cwd=ROOT, stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0 and res.stdout.rstrip().endswith("ok"), res.stdout


@pytest.mark.gpu
def test_several_threads_at_once():
    """Four threads with a stream each make whole calls on lists that share a plan."""
    if q._pylist is None:
        pytest.skip("torchft_amd._pylist is not built")
    g = torch.Generator("cuda").manual_seed(5)
    lists = [[torch.randn(40, 130, generator=g, device="cuda"), torch.randn(9, 64, generator=g, device="cuda")] for _ in range(4)]

    def one_pass(ts, quantize):
        ts = [t.clone() for t in ts]
        packed = quantize(ts)
        torchft_amd.fused_reduce_fp8(ts, packed, 2, 1, ReduceOp.AVG)
        torchft_amd.fused_dequantize_from_fp8(ts, packed, 2)
        return [packed, *ts]

    def named(ts):
        return torchft_amd.fused_quantize_into_fp8(ts, 2)

    want = [one_pass(ts, named) for ts in lists]
    torch.cuda.synchronize()
    failed, start = [], threading.Barrier(len(lists))

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait(30)
                for k in range(100):
                    got = one_pass(lists[i], named if k % 2 else lambda ts: torchft_amd.prepare(ts, 2).quantize())
                    assert all(torch.equal(a, b) for a, b in zip(got, want[i])), k
        except BaseException as exc:
            failed.append((i, exc))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(lists))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed and not any(t.is_alive() for t in threads), failed
