"""The block GEMM of msq_moe_prefill with every number of token tiles an item can have, each full, one short of full and
with one entry in its last tile; one block of K (nothing to fetch ahead) and several, an odd and an even number."""
import pytest

import oracle as O
import test_moe_prefill_gpu as P

pytestmark = pytest.mark.gpu

SIZES = [113, 112, 111, 97, 96, 81, 80, 65, 64, 49, 48, 47, 33, 32, 17, 16, 1]


@pytest.mark.parametrize("t", [O.IQ1_S, O.IQ2_XXS], ids=["IQ1_S", "IQ2_XXS"])
@pytest.mark.parametrize("dim,inter", [(256, 512), (768, 256), (1024, 768)])
def test_every_number_of_token_tiles(dev, monkeypatch, t, dim, inter):
    n, k = max(SIZES), len(SIZES)
    monkeypatch.setattr(P, "make_routing", lambda *_: [[e for e in range(k) if i < SIZES[e]] for i in range(n)])
    c = P.build(t, t, O.Q6_K, n, k, k, False, "", dim, inter)
    y, same = P.run_gpu(c)
    err_h, err_f, _ = P.check(c, y, 0)
    assert same and err_h <= 1e-3 and err_f <= 5e-3  # the bounds of test_moe_prefill_gpu.py (the reference's)


@pytest.mark.parametrize("t", [O.IQ1_S, O.IQ2_XXS], ids=["IQ1_S", "IQ2_XXS"])
@pytest.mark.parametrize("dim,inter,small", [(256, 4096, 14), (8192, 256, 87)])
def test_more_units_than_workgroups(dev, monkeypatch, t, dim, inter, small):
    """Workgroups that take unit after unit, of every number of token tiles: both sizes of items have more units than the
    chip holds workgroups, in the first product (4096 rows; a shared expert beside it) and in the second (8192: row chunks in
    pairs)."""
    sizes = SIZES + [15, 1] * (small // 2) + [2] * (small % 2)
    n, k = 224, 8
    routes = [[] for _ in range(n)]
    for e, m in enumerate(sizes):
        for i in sorted(range(n), key=lambda i: (len(routes[i]), (i + 37 * e) % n))[:m]:
            routes[i].append(e)
    monkeypatch.setattr(P, "make_routing", lambda *_: routes)
    c = P.build(t, t, O.Q6_K, n, k, len(sizes), dim == 256, "", dim, inter)
    y, same = P.run_gpu(c)
    err_h, err_f, _ = P.check(c, y, 0)
    assert same and err_h <= 1e-3 and err_f <= 5e-3  # the bounds of test_moe_prefill_gpu.py (the reference's)


@pytest.mark.parametrize("entries", [1, 39, 40, 41])
def test_rows_by_entry_and_by_token(dev, monkeypatch, entries):
    """Fewer entries than the 40 tokens: their rows are gathered; as many and more: found by the token."""
    n, k = 40, 2
    monkeypatch.setattr(P, "make_routing", lambda *_: [[0] * (i < entries) + [1] * (n + i < entries) for i in range(n - 1, -1, -1)])
    c = P.build(O.IQ2_XXS, O.IQ1_S, O.Q6_K, n, k, 2, False, "", 512, 256)
    y, same = P.run_gpu(c)
    err_h, err_f, _ = P.check(c, y, 0)
    assert same and err_h <= 1e-3 and err_f <= 5e-3  # the bounds of test_moe_prefill_gpu.py (the reference's)
