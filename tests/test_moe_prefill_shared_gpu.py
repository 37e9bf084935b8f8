"""The dense kernel of a Q6_K / Q8_0 shared expert in msq_moe_prefill at the edges of its tiles: one token, one short of /
exactly / one past a 128-token block, the smallest matrices, rows of 64 x an odd number of chunks, one and several blocks
of K, with and without routed experts beside it."""
import pytest

import oracle as O
from test_moe_prefill_gpu import build, check, run_gpu

pytestmark = pytest.mark.gpu

CASES = [  # (shared type, n, k, n_exp, dim, inter)
    (O.Q6_K, 1, 1, 2, 256, 256), (O.Q8_0, 1, 1, 2, 256, 256), (O.Q6_K, 127, 1, 3, 512, 256), (O.Q8_0, 128, 1, 3, 256, 768),
    (O.Q6_K, 129, 1, 3, 256, 512), (O.Q8_0, 257, 1, 3, 512, 256), (O.Q6_K, 17, 2, 4, 1280, 768), (O.Q8_0, 100, 2, 4, 768, 1280),
]


@pytest.mark.parametrize("sh,n,k,n_exp,dim,inter", CASES, ids=lambda v: None)
def test_shared_expert_tile_kernel(dev, sh, n, k, n_exp, dim, inter):
    c = build(O.IQ2_XXS, O.IQ1_S, sh, n, k, n_exp, True, "zipf:0.8", dim, inter)
    y, same = run_gpu(c)
    err_h, err_f, _ = check(c, y, 0)
    assert same and err_h <= 1e-3 and err_f <= 5e-3  # the bounds of test_moe_prefill_gpu.py (the reference's)
