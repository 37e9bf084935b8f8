"""Few-token kernel up to 2048 columns: workgroups of one row tile meet tile by tile, of more two tiles at a time; each on either side
of that line, a workgroup of a single wave, and the format and token counts that keep two."""
import pytest

import oracle as O
from test_matmul_rows_gpu import test_matmul_of_little_work as matmul
from test_matvec_n_rows_gpu import test_few_token_kernel_vs_oracle as matvec_n

N_CASES = [  # (type, rows, cols, groups, n, accumulate)
    (O.Q6_K, 4096, 1280, 1, 16, True), (O.Q6_K, 20000, 1280, 1, 16, False), (O.IQ4_NL, 4096, 1280, 1, 8, False), (O.IQ4_NL, 4096, 1280, 1, 9, True),
    (O.IQ2_XXS, 2064, 256, 1, 8, False), (O.Q5_K, 30000, 256, 1, 5, True), (O.IQ1_S, 4096, 2048, 1, 12, False), (O.IQ1_S, 4112, 2048, 1, 12, False),
    (O.Q6_K, 8192, 1024, 8, 7, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("t,rows,cols,groups,n,acc", N_CASES, ids=lambda v: None)
def test_matvec_n_meetings(dev, t, rows, cols, groups, n, acc):
    matvec_n(dev, t, rows, cols, groups, n, acc)


@pytest.mark.gpu
@pytest.mark.parametrize("t,rows,cols,n,acc,xs", [(O.IQ4_NL, 1024, 2048, 100, False, 2048), (O.Q6_K, 2000, 1024, 40, True, 0), (O.IQ1_S, 1100, 768, 150, False, 0),
                                                  (O.Q6_K, 1024, 2048, 130, True, 0)], ids=lambda v: None)
def test_matmul_meetings(dev, t, rows, cols, n, acc, xs):
    matmul(dev, t, rows, cols, n, acc, xs)
