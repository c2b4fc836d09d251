"""Every variant of the kernels of quantize's second launch against the CPU checker, by bytes."""

import os
import subprocess

import pytest
import torch

from test_gpu_columns import transposed
from test_gpu_parity import NT, q, same_bytes  # noqa: F401 (q is a fixture)

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# (slots, rows and columns): lists that between them take every variant; which ones, the test below says
HALF = [
    (3, [(13, 5292), (9, 2210), (41, 41), (18, 1040)]),
    (8, [(11, 685), (636, 73), (6919, 18), (12, 1145), (23, 602), (12, 6235), (927, 30), (9, 3731), (166, 26),
         (201, 34), (939, 44), (744, 33)]),
    (3, [(34, 18), (11, 1373), (41, 29), (9, 2748)]),
    (3, [(12, 2132), (94, 113), (10, 8702), (56, 96), (19, 37), (32, 1762)]),
    (1, [(223, 147), (13, 3466), (27, 2031), (28, 572), (3835, 17)]),
    (8, [(879, 19), (10, 27), (9, 8410)]),
    (8, [(11, 12550), (9, 5261)]),
    (8, [(753, 98), (1192, 28), (33, 474), (31, 282), (15, 3928), (21, 120), (22, 3311), (42, 19), (117, 189),
         (47, 344), (113, 280), (11, 34), (121, 235), (1260, 177)]),
    (8, [(15, 4103), (1532, 56), (1342, 78), (21, 12490), (923, 266), (471, 274), (169, 2064), (19, 7164), (27, 62),
         (16, 9455), (138, 962), (350, 899), (54, 355), (31, 130), (30, 113)]),
    (8, [(19, 6478), (11, 7763), (17, 11280), (1005, 156), (12, 2826)]),
    (8, [(144, 873), (2077, 34), (67, 1037), (13, 136), (41, 435), (166, 3122), (9, 573), (177, 55), (23, 1324),
         (2578, 199), (262, 53), (16209, 29), (61, 31), (322, 408), (763, 1156), (67, 49)]),
    (8, [(25, 1872), (9, 474), (4944, 80), (391, 104), (48, 176), (9, 8245), (168, 225), (14, 33), (898, 84),
         (169, 1198), (31, 345), (12, 9888), (1031, 91), (14, 5047), (754, 237), (22, 23), (44, 2542), (64, 213),
         (31, 8252)]),
    (8, [(21, 1953), (23, 22), (76, 24), (15, 572), (21, 2822), (149, 2848), (200, 172), (3938, 280), (41, 130),
         (31, 457), (15, 3693), (8105, 47), (4784, 69), (41, 197), (14, 1013), (1883, 20), (37, 4045), (1276, 1120),
         (134, 74), (438, 370), (1502, 41), (9, 2920)]),
    (8, [(44, 2878), (1381, 413), (63, 171), (166960, 17), (784, 513), (44, 417)]),
    (8, [(5921, 4165)]),
]
FULL = [
    (8, [(95, 119), (11, 1197), (22, 2375), (126, 807), (9, 9826), (187, 163)]),
    (3, [(13, 5292), (9, 2210), (41, 41), (18, 1040)]),
    (1, [(17, 2200), (10, 1300), (13, 46)]),
    (8, [(3169, 35), (283, 45), (9, 7096), (56, 1180)]),
    (3, [(11, 12496), (9, 9300)]),
    (8, [(10, 13457), (14, 41), (11, 139), (430, 237)]),
    (1, [(25, 39), (31, 102), (166, 1104), (231, 193), (10, 734), (76, 845), (2242, 338), (74, 789), (19, 1611),
         (25, 527), (234, 287), (5911, 35), (459, 97), (293, 42), (500, 509)]),
    (8, [(89, 2930), (689, 255), (9, 13755), (518, 81), (9, 5278), (221, 223), (325, 840), (198, 283), (41, 23),
         (829, 42), (84, 755), (1072, 118), (239, 900), (652, 207), (93, 1799)]),
    (3, [(16, 1687), (205, 672), (31, 21), (8630, 274), (93, 843), (179, 1126)]),
    (8, [(72, 13080), (12, 262), (593, 62), (425, 301), (1152, 22), (426, 30)]),
    (8, [(3054, 4137)]),
]


def expected(half):
    """kernel/groups/steps that a variant holds; 16: rows of more than 12."""
    any4 = {f"any4/{g}/{s}" for g in (2, 4, 8, 16) for s in (1, 2, 4)} | {"any4/32/1"}
    any12 = {w.replace("any4", "any12") for w in any4} | {"any12/2/8", "any12/2/12", "any12/2/16", "any12/4/12"}
    two = {f"two12/2/{s}" for s in (1, 2, 4, 8, 12, 16)}
    few = {f"two4/2/{s}" for s in (1, 2, 4)} | {f"two8/2/{s}" for s in (1, 2, 4, 8)}
    return any4 | any12 | two | (few if half else set())


@pytest.mark.parametrize("dtype, lists, half", [(0, FULL, False), (1, HALF, True), (2, HALF, True)])
def test_the_lists_reach_every_variant(tmp_path, dtype, lists, half):
    exe = str(tmp_path / "column_kernels")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-o", exe, os.path.join(HERE, "column_kernels.cpp"),
                           os.path.join(ROOT, "torchft_amd", "csrc", "tftq_plan.cpp")])
    lines = "".join(f"{dtype} {ws} " + " ".join(f"{m} {n}" for m, n in shapes) + "\n" for ws, shapes in lists)
    res = subprocess.run([exe], input=lines, stdout=subprocess.PIPE, text=True, timeout=60)
    assert res.returncode == 0 and set(res.stdout.split()) == expected(half)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, lists", [(torch.float32, FULL), (torch.float16, HALF), (torch.bfloat16, HALF)])
def test_every_variant(q, oracle, dtype, lists):  # noqa: F811
    for ws, shapes in lists:
        g = torch.Generator().manual_seed(ws)
        views, bases = zip(*[transposed(m, n, 0, 0, dtype, g) for m, n in shapes])
        packed = oracle.fused_quantize_into_fp8([v.clone() for v in views], ws, nthreads=NT)
        gpu = [torch.as_strided(b.cuda(), v.shape, v.stride(), 0) for v, b in zip(views, bases)]
        same_bytes(q.fused_quantize_into_fp8(gpu, ws), packed, f"{ws} slots, {shapes}")
