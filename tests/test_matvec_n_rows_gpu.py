"""The few-token matrix-core kernel of msq_matvec_n (three tokens and more of the block formats) at the edges of its
shapes: ragged last row tiles, groups, one / two weight stages per wave, rows that end with half a stage, one tile and
several tiles per workgroup, 8 / 9 / 16 tokens, accumulation, weights off 16-byte boundaries."""
import numpy as np
import pytest

import oracle as O
from macseek_amd import quant as q
from util import place_in_arena, up

pytestmark = pytest.mark.gpu

CASES = [  # (type, rows, cols, groups, n, accumulate)
    (O.Q6_K, 257, 256, 1, 3, False), (O.Q6_K, 300, 2048, 1, 8, True), (O.Q6_K, 1040, 2304, 1, 9, False),
    (O.Q6_K, 1024, 4096, 8, 16, False), (O.Q6_K, 1031, 4352, 1, 16, True), (O.Q6_K, 8208, 256, 1, 7, False),
    (O.Q6_K, 16400, 512, 1, 2, False), (O.Q5_K, 272, 1280, 1, 5, True), (O.Q5_K, 1056, 8192, 1, 11, False),
    (O.Q5_K, 12301, 256, 1, 16, False), (O.IQ4_NL, 260, 128, 1, 3, False), (O.IQ4_NL, 777, 1152, 1, 9, True),
    (O.IQ4_NL, 1536, 4224, 1, 10, False), (O.IQ4_NL, 512, 640, 2, 4, False), (O.IQ1_S, 513, 768, 1, 3, False),
    (O.IQ1_S, 1100, 5120, 1, 16, True), (O.IQ1_S, 300, 4096, 1, 12, False), (O.IQ2_XXS, 305, 1024, 1, 8, True),
    (O.IQ2_XXS, 1024, 7936, 1, 6, False), (O.IQ2_XXS, 1280, 512, 4, 13, False),
]


@pytest.mark.parametrize("t,rows,cols,groups,n,acc", CASES, ids=lambda v: None)
def test_few_token_kernel_vs_oracle(dev, t, rows, cols, groups, n, acc):
    Wb = O.random_blocks(t, rows * cols, 5 + rows)
    xs = cols * groups
    X, Y0 = O.randn(xs * n, 6 + n), O.randn(rows * n, 7)
    _, (W,) = place_in_arena([Wb])
    Xd, Yd = up(X), up(np.concatenate([Y0, np.full(64, 3.0, np.float32)]))
    e = q.Enc()
    q.encode_matvec_n(e, t, W, rows, cols, q.Buffer.of(Xd), q.Buffer.of(Yd), n, acc, groups)
    e.wait()
    got = Yd.cpu().numpy()
    assert (got[rows * n:] == 3.0).all()
    Xh = X.astype(np.float16).astype(np.float32)  # the kernel's staging: exact payloads, fp32 scales and sums
    for tok in range(n):
        ry, mag, _ = O.matvec(t, Wb, rows, cols, Xh[tok * xs:(tok + 1) * xs], groups)
        if acc:
            y0 = Y0[tok * rows:(tok + 1) * rows].astype(np.float64)
            ry, mag = ry + y0, mag + np.abs(y0)
        d = np.abs(got[tok * rows:(tok + 1) * rows] - ry) / (mag + 1e-12)
        # fp32 sums of at most 8192 products: a few units of 2^-24 of the sum of magnitudes (the reference's bound)
        assert float(np.max(d)) <= 2e-6
