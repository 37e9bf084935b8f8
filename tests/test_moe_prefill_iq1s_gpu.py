"""IQ1_S experts in msq_moe_prefill, whose block bytes reach the matrix cores through LDS: one block of K and several, a
last row chunk that is not full, one to three token tiles, popular experts of 49 entries and of more than 112."""
import pytest

import oracle as O
from test_moe_prefill_gpu import build, check, run_gpu

pytestmark = pytest.mark.gpu

CASES = [  # (n, k, n_exp, dim, inter)
    (1, 1, 1, 256, 256), (16, 1, 1, 256, 512), (17, 1, 1, 768, 256), (48, 1, 1, 512, 1280), (49, 1, 1, 1280, 512),
    (112, 1, 1, 256, 256), (113, 1, 1, 512, 768), (60, 3, 5, 2304, 1280),
]


@pytest.mark.parametrize("n,k,n_exp,dim,inter", CASES, ids=lambda v: None)
def test_iq1s_experts_through_lds(dev, n, k, n_exp, dim, inter):
    c = build(O.IQ1_S, O.IQ1_S, O.IQ1_S, n, k, n_exp, n > 40, "zipf:0.8", dim, inter)
    y, same = run_gpu(c)
    err_h, err_f, _ = check(c, y, 0)
    assert same and err_h <= 1e-3 and err_f <= 5e-3  # the bounds of test_moe_prefill_gpu.py (the reference's)
