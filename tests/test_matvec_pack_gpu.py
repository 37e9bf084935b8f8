"""Decode matvec, several matrix rows as one launched row: two, four and eight of them, sums of 16 and of 8 lanes, whole and partly
idle waves, numbers of rows that only allow fewer, a ragged last tile, weight rows through LDS, a second workgroup per CU, either
prologue of a fused norm, accumulation."""
import numpy as np
import pytest
import torch

import oracle as O
from macseek_amd import quant as q
from test_matvec_rmsnorm_gpu import test_fused_equals_norm_then_matvec_and_oracle as with_norm
from util import TOL_NORTH_STAR, matvec_errors, place_in_arena, tol_ref, up

pytestmark = pytest.mark.gpu

CASES = [  # (type, rows, cols)
    (O.Q6_K, 32776, 256), (O.Q5_K, 8196, 512), (O.Q6_K, 32768, 512), (O.Q8_0, 6002, 512), (O.Q5_K, 9000, 768), (O.Q6_K, 20002, 768),
    (O.Q6_K, 8200, 1280), (O.Q5_K, 16392, 1280), (O.Q6_K, 25600, 1280), (O.Q8_0, 12288, 1280), (O.Q8_0, 20000, 1280), (O.Q6_K, 4100, 1536), (O.Q8_0, 32772, 1536),
    (O.Q5_K, 4104, 2304), (O.Q6_K, 7002, 2304), (O.Q6_K, 4100, 2560), (O.Q5_K, 12004, 2560), (O.F32, 2100, 384 * 2), (O.BF16, 5002, 1280),
    (O.Q6_K, 5000, 5120),
]


@pytest.mark.parametrize("acc", [False, True])
@pytest.mark.parametrize("t,rows,cols", CASES, ids=lambda v: None)
def test_packed_rows_vs_oracle(dev, t, rows, cols, acc):
    Wb = O.random_blocks(t, rows * cols, 7 + cols, 0.03)
    x, y0 = O.randn(cols, 5), O.randn(rows, 6)
    _, (W,) = place_in_arena([Wb])
    xd, yd = up(x), up(np.concatenate([y0, np.full(64, 3.0, np.float32)]))
    e = q.Enc()
    q.encode_matvec(e, t, W, rows, cols, q.Buffer.of(xd), q.Buffer.of(yd), acc)
    e.wait()
    got = yd.cpu().numpy()
    assert (got[rows:] == 3.0).all()
    ry, mag, wn2 = O.matvec(t, Wb, rows, cols, x)
    if acc:
        assert float(np.max(np.abs(got[:rows] - (ry + y0)) / (mag + np.abs(y0) + 1e-12))) <= tol_ref(t, cols)
    else:
        err_ref, err_ns = matvec_errors(got[:rows], ry, mag, wn2, x, rows, cols, 1)
        assert err_ns <= TOL_NORTH_STAR and err_ref <= tol_ref(t, cols)


@pytest.mark.parametrize("t,rows,cols", [(O.Q6_K, 32776, 256), (O.Q5_K, 8196, 512), (O.Q6_K, 9000, 768), (O.Q6_K, 25600, 1280), (O.Q5_K, 30720, 1280),
                                         (O.Q8_0, 16392, 1280), (O.Q6_K, 12004, 2560), (O.Q5_K, 8008, 2304)], ids=lambda v: None)
def test_packed_rows_with_norm(dev, t, rows, cols):
    with_norm(dev, t, rows, cols)


@pytest.mark.parametrize("t,rows,cols", [(O.Q6_K, 32768, 1280), (O.Q5_K, 8196, 512), (O.Q6_K, 9000, 768), (O.Q5_K, 8008, 2304), (O.Q8_0, 20000, 1280),
                                         (O.Q6_K, 32776, 256), (O.Q6_K, 4100, 1536), (O.Q8_0, 32772, 768)], ids=lambda v: None)
def test_packed_rows_have_the_bits_of_chunks(dev, t, rows, cols):
    # chunks launched with matvec_cfg's shape go row by row, the whole matrix packed: sums of 16 and of 8 lanes
    Wd, xd = up(O.random_blocks(t, rows * cols, 11 + cols)), up(O.randn(cols, 12))
    W, rb, cfg = q.Buffer.of(Wd), q.row_bytes(t, cols), q.matvec_cfg(t, rows, cols)
    full, parts = torch.empty(rows, device=dev), torch.empty(rows, device=dev)
    e = q.Enc()
    q.encode_matvec(e, t, W, rows, cols, q.Buffer.of(xd), q.Buffer.of(full))
    chunk = cfg.nr * cfg.rsg * 37
    for r0 in range(0, rows, chunk):
        n = min(chunk, rows - r0)
        q.encode_matvec(e, t, W.sub(r0 * rb, n * rb), n, cols, q.Buffer.of(xd), q.Buffer.of(parts).sub(r0 * 4, n * 4), False, 1, cfg)
    e.wait()
    assert torch.equal(full, parts)
