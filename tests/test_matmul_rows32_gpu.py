"""The few-token kernel of msq_matmul in blocks of 32 tokens: one, a ragged and several blocks, one row tile and several per
workgroup (also an odd number where two meet at a time), a ragged last tile, rows in two launches (with half a weight stage at
the end), fp32 and strided fp16 activations, overwriting and accumulating; and, on the CPU, both sides of the rule's lines."""
import pytest

import oracle as O
from test_matmul_rows_gpu import FEW, FUSED, GEMM, TILE, route, test_matmul_of_little_work as check

CASES = [  # (type, rows, cols, n, accumulate, fp16 activations' row stride or 0)
    (O.IQ4_NL, 1537, 4096, 33, False, 0), (O.Q6_K, 1540, 4096, 256, True, 0), (O.Q5_K, 1153, 3840, 200, False, 3844),
    (O.IQ1_S, 2048, 2304, 129, True, 0), (O.IQ2_XXS, 8200, 4096, 17, False, 0), (O.IQ2_XXS, 16400, 1280, 64, True, 1284),
    (O.Q6_K, 16384, 1536, 40, False, 1536), (O.Q5_K, 20000, 1280, 31, True, 0), (O.IQ4_NL, 16384, 1664, 100, False, 0),
    (O.IQ4_NL, 5130, 7808, 50, True, 7808), (O.IQ4_NL, 5130, 6272, 19, False, 0), (O.IQ2_XXS, 5120, 8192, 64, True, 0),
    (O.Q6_K, 6150, 7168, 32, True, 0), (O.Q5_K, 6144, 6144, 18, False, 6148), (O.IQ1_S, 5121, 6400, 41, False, 0),
    (O.Q6_K, 1030, 768, 700, False, 0), (O.IQ1_S, 3000, 1024, 200, True, 0), (O.IQ2_XXS, 1024, 512, 900, False, 512),
]

ROUTES = [  # as in test_matmul_rows_gpu.py
    ((O.IQ4_NL, 16384, 1536, 32, 0, 0), FEW), ((O.IQ4_NL, 16384, 1536, 33, 0, 0), FUSED), ((O.IQ4_NL, 16384, 1536, 40, 0, 0), FEW),
    ((O.IQ4_NL, 16384, 1536, 128, 0, 0), FEW), ((O.IQ4_NL, 16384, 1536, 129, 0, 0), TILE), ((O.IQ4_NL, 20000, 1536, 100, 0, 0), TILE),
    ((O.IQ4_NL, 16384, 1280, 100, 0, 0), TILE), ((O.IQ2_XXS, 16384, 1536, 64, 0, 0), FEW), ((O.IQ2_XXS, 16384, 1536, 65, 0, 0), TILE),
    ((O.Q6_K, 16384, 1024, 20, 0, 0), FUSED), ((O.Q6_K, 16384, 1280, 20, 0, 0), FEW), ((O.Q6_K, 65536, 1280, 20, 0, 0), FEW),
    ((O.Q6_K, 65552, 1280, 20, 0, 0), FUSED), ((O.IQ1_S, 16384, 1280, 20, 0, 0), FEW), ((O.IQ1_S, 16400, 1280, 20, 0, 0), FUSED),
    ((O.Q5_K, 8192, 2048, 47, 0, 0), FUSED), ((O.Q5_K, 8192, 2048, 48, 0, 0), FEW), ((O.Q6_K, 8192, 3584, 100, 0, 0), FEW),
    ((O.Q6_K, 8192, 3328, 100, 0, 0), FUSED), ((O.Q5_K, 8192, 3840, 100, 0, 0), FUSED), ((O.Q5_K, 8192, 4096, 100, 0, 0), FEW),
    ((O.IQ4_NL, 5120, 8192, 20, 0, 0), FEW), ((O.IQ4_NL, 5119, 8192, 20, 0, 0), FUSED),
    ((O.IQ4_NL, 5120, 8320, 20, 0, 0), FUSED), ((O.IQ4_NL, 5120, 5888, 20, 0, 0), FUSED), ((O.Q6_K, 6144, 8192, 32, 0, 0), FEW),
    ((O.Q6_K, 6144, 8192, 40, 0, 0), FUSED), ((O.Q6_K, 5888, 8192, 32, 0, 0), FUSED), ((O.IQ1_S, 5120, 8192, 32, 0, 0), FUSED),
    ((O.IQ1_S, 5120, 8192, 64, 0, 0), FEW), ((O.IQ1_S, 5120, 8192, 64, 1, 0), FUSED), ((O.IQ2_XXS, 1152, 4096, 256, 0, 0), FEW),
    ((O.IQ2_XXS, 1136, 4096, 256, 0, 0), FUSED), ((O.IQ2_XXS, 2048, 4096, 256, 0, 0), FEW), ((O.IQ2_XXS, 2064, 4096, 256, 0, 0), GEMM),
    ((O.Q6_K, 16384, 1536, 40, 1, 1538), FUSED),
]

LOSING = [  # the fused kernel is ahead: fp16 Q6_K in the first half of 4096 rows, two launches that have just begun another round of workgroups
    ((O.Q6_K, 16384, 1280, 45, 1, 0), FEW), ((O.Q6_K, 16385, 1280, 45, 1, 0), FUSED), ((O.Q6_K, 18432, 1536, 40, 1, 0), FUSED),
    ((O.Q6_K, 18433, 1536, 40, 1, 0), FEW), ((O.Q6_K, 20481, 1280, 48, 1, 0), FUSED), ((O.Q6_K, 20481, 1280, 49, 1, 0), FEW),
    ((O.Q6_K, 20481, 1280, 48, 0, 0), FEW), ((O.Q6_K, 16385, 1792, 45, 1, 0), FEW), ((O.Q6_K, 18432, 1280, 32, 1, 0), FEW),
    ((O.IQ2_XXS, 5440, 7424, 44, 1, 0), FUSED), ((O.IQ2_XXS, 5441, 7424, 44, 1, 0), FEW), ((O.IQ2_XXS, 5180, 7680, 44, 1, 0), FEW),
    ((O.IQ2_XXS, 5180, 7424, 32, 1, 0), FEW), ((O.IQ2_XXS, 5180, 6656, 48, 0, 0), FUSED), ((O.IQ2_XXS, 5180, 6656, 49, 0, 0), FEW),
    ((O.IQ2_XXS, 6144, 6400, 60, 0, 0), FEW), ((O.IQ2_XXS, 6145, 6400, 60, 0, 0), FUSED), ((O.IQ2_XXS, 6512, 6400, 60, 0, 0), FUSED),
    ((O.IQ2_XXS, 6513, 6400, 60, 0, 0), FEW), ((O.IQ4_NL, 5200, 6528, 20, 0, 0), FUSED), ((O.IQ4_NL, 5441, 6528, 20, 0, 0), FEW),
    ((O.IQ4_NL, 5200, 6656, 20, 0, 0), FEW), ((O.Q5_K, 6144, 6656, 20, 0, 0), FUSED), ((O.Q5_K, 6144, 6656, 20, 1, 0), FEW),
    ((O.Q5_K, 6513, 6656, 20, 0, 0), FEW), ((O.Q6_K, 6144, 6656, 20, 0, 0), FEW),
]


def test_which_calls_it_serves():
    assert [(c, route(*c)) for c, _ in ROUTES] == ROUTES


def test_which_calls_it_leaves_to_the_fused_kernel():
    assert [(c, route(*c)) for c, _ in LOSING] == LOSING


@pytest.mark.gpu
@pytest.mark.parametrize("t,rows,cols,n,acc,xs", CASES, ids=lambda v: None)
def test_blocks_of_32_tokens(dev, t, rows, cols, n, acc, xs):
    check(dev, t, rows, cols, n, acc, xs)
