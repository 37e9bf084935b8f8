"""msq_matmul / msq_matmul_h calls of little work over block formats: the few-token kernel in blocks of sixteen tokens. Ragged
last token block and last row tile, one and several row tiles per workgroup, half a weight stage at the end of a row, fp16
activations with a stride, both sides of the switch to the other kernels."""
import numpy as np
import pytest
import torch

import oracle as O
from macseek_amd import quant as q
from test_matmul_gpu import reference
from util import place_in_arena, up

pytestmark = pytest.mark.gpu

CASES = [  # (type, rows, cols, n, accumulate, fp16 activations' row stride or 0)
    (O.IQ4_NL, 577, 640, 17, False, 0), (O.IQ4_NL, 100, 4096, 100, True, 4104), (O.Q6_K, 1040, 256, 33, False, 0),
    (O.Q6_K, 250, 2304, 31, True, 2308), (O.Q5_K, 16, 512, 1000, False, 0), (O.Q5_K, 1030, 1280, 97, True, 1280),
    (O.IQ1_S, 2000, 2048, 47, False, 2048), (O.IQ1_S, 5, 4096, 18, True, 0), (O.IQ2_XXS, 777, 3840, 64, False, 0),
    (O.IQ2_XXS, 1024, 2048, 513, True, 0), (O.IQ2_XXS, 1024, 2048, 512, False, 2052), (O.Q6_K, 8192, 256, 20, False, 0),
]


@pytest.mark.parametrize("t,rows,cols,n,acc,xs", CASES, ids=lambda v: None)
def test_matmul_of_little_work(dev, t, rows, cols, n, acc, xs):
    Wb = O.random_blocks(t, rows * cols, 5 + rows)
    X, Y0 = O.randn(n * cols, 13 + n), O.randn(n * rows, 14)
    _, (W,) = place_in_arena([Wb], first=16, gap=16)
    Yd = up(Y0.copy())
    e = q.Enc()
    if xs:
        X16 = torch.full((n, xs), 7.0, dtype=torch.float16, device=dev)
        X16[:, :cols] = up(X.astype(np.float16)).view(n, cols)
        q.encode_matmul_h(e, t, W, rows, cols, q.Buffer.of(X16), q.Buffer.of(Yd), n, acc, xs)
    else:
        Xd = up(X)
        q.encode_matmul(e, t, W, rows, cols, q.Buffer.of(Xd), q.Buffer.of(Yd), n, acc)
    e.wait()
    got = Yd.cpu().numpy().astype(np.float64).reshape(n, rows)
    sh, _, mag, _ = reference(t, Wb, rows, cols, X, n)
    base = Y0.reshape(n, rows).astype(np.float64) if acc else 0.0
    assert float(np.max(np.abs(got - (sh + base)) / (mag + np.abs(base) + 1e-12))) <= 1e-5  # the bound of test_matmul_gpu.py
