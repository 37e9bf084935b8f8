"""A Q6_K / Q8_0 shared expert over few tokens in msq_moe_prefill (the few-token kernel): one token, both sides of a block of sixteen
and of the lines to the tile kernel (112 tokens, few experts one of which has more than 48 entries), one weight stage a row, an odd number of them over waves of two, the longest
rows, rows too long for the LDS (Q8_0: the tile kernel stays), a ragged number of row tiles per workgroup."""
import pytest

import oracle as O
from test_moe_prefill_gpu import build, check, run_gpu

pytestmark = pytest.mark.gpu

CASES = [  # (shared type, n, k, n_exp, dim, inter)
    (O.Q6_K, 2, 1, 2, 256, 256), (O.Q8_0, 16, 1, 3, 512, 256), (O.Q6_K, 17, 1, 3, 4352, 256), (O.Q8_0, 15, 1, 3, 4352, 512),
    (O.Q6_K, 33, 1, 3, 768, 4352), (O.Q8_0, 20, 1, 3, 512, 4352), (O.Q6_K, 112, 2, 4, 1024, 768), (O.Q8_0, 113, 2, 4, 1024, 768),
    (O.Q6_K, 3, 1, 2, 8192, 512), (O.Q8_0, 3, 1, 2, 6656, 256), (O.Q8_0, 3, 1, 2, 7168, 256), (O.Q6_K, 40, 1, 3, 2560, 2304),
]


@pytest.mark.parametrize("sh,n,k,n_exp,dim,inter", CASES, ids=lambda v: None)
def test_shared_expert_few_tokens(dev, sh, n, k, n_exp, dim, inter):
    c = build(O.IQ2_XXS, O.IQ1_S, sh, n, k, n_exp, True, "zipf:0.8", dim, inter)
    y, same = run_gpu(c, n % 2 == 1)
    err_h, err_f, _ = check(c, y, 0, n % 2 == 1)
    assert same and err_h <= 1e-3 and err_f <= 5e-3  # the bounds of test_moe_prefill_gpu.py (the reference's)


@pytest.mark.parametrize("sh,n,k,n_exp,kind", [(O.Q6_K, 112, 1, 4, "zipf:0"), (O.Q8_0, 112, 2, 6, "zipf:0"), (O.Q6_K, 48, 2, 3, "popular"),
                                               (O.Q6_K, 49, 2, 3, "popular"), (O.Q8_0, 49, 2, 3, "popular")], ids=lambda v: None)
def test_both_sides_of_a_crowded_expert(dev, sh, n, k, n_exp, kind):
    c = build(O.IQ1_S, O.IQ2_XXS, sh, n, k, n_exp, True, kind, 1024, 768)
    entries = [b - a for a, b in zip(c["offs"], c["offs"][1:])]
    assert (max(entries) > 48) == (n == 49)
    y, same = run_gpu(c)
    err_h, err_f, _ = check(c, y, 0, False)
    assert same and err_h <= 1e-3 and err_f <= 5e-3
