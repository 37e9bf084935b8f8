"""GPU tests of msq_rmsnorm and msq_matvec_rmsnorm (the decode matvec with the input RMSNorm fused in).

Mirrors the reference's tests/test_dec_fuse.mm:27-53: the fused call must equal rmsnorm -> matvec bit for bit, on its
six cases plus the BASELINE shapes; and, since that identity alone would also hold for two wrong kernels, both are
compared with the CPU oracle (norm in double; double dot of the normalized row).
"""
import numpy as np
import pytest
import torch

import oracle as O
from macseek_amd import arch, quant as q
from util import TOL_NORTH_STAR, matvec_errors, place_in_arena, tol_ref, up

pytestmark = pytest.mark.gpu

CASES = [  # tests/test_dec_fuse.mm:30-31, then the attention-projection shapes of BASELINE configs[4] and edge shapes
    (O.Q6_K, 32768, 1280), (O.Q5_K, 32768, 1280), (O.BF16, 4096, 1280), (O.Q8_0, 1000, 2048), (O.F32, 77, 1536),
    (O.Q6_K, 300, 5120),
    (O.Q6_K, 1536, 7168), (O.Q5_K, 512, 7168), (O.IQ4_NL, 7168, 4096), (O.BF16, 384, 7168), (O.F16, 40, 256),
    (O.Q8_0, 5000, 1024), (O.Q6_K, 64, 14336),
]


@pytest.mark.parametrize("t,rows,cols", CASES, ids=lambda v: None)
def test_fused_equals_norm_then_matvec_and_oracle(dev, t, rows, cols):
    eps = 1e-20 if rows % 2 else 1e-6
    Wb = O.random_blocks(t, rows * cols, 11 + cols, 0.03)
    x = (O.randn(cols, 5) * 3.0).astype(np.float32)
    nw = (1.0 + 0.2 * O.randn(cols, 6)).astype(np.float32)
    arena, (W,) = place_in_arena([Wb])
    xd, nwd = up(x), up(nw)
    xn = torch.zeros(cols, dtype=torch.float32, device=dev)
    y0 = torch.zeros(rows, dtype=torch.float32, device=dev)
    y1 = torch.full((rows + 8,), 4.0, dtype=torch.float32, device=dev)
    e = q.Enc()
    arch.encode_rmsnorm(e, q.Buffer.of(xd), q.Buffer.of(nwd), q.Buffer.of(xn), 1, cols, eps)
    e.barrier()
    q.encode_matvec(e, t, W, rows, cols, q.Buffer.of(xn), q.Buffer.of(y0))
    q.encode_matvec_rmsnorm(e, t, W, rows, cols, q.Buffer.of(xd), q.Buffer.of(nwd), eps, q.Buffer.of(y1))
    e.wait()
    assert torch.equal(y0, y1[:rows]) and bool((y1[rows:] == 4.0).all())        # bit for bit; nothing past the rows
    # the norm against the oracle (float reduction against double: a few ulp)
    xn_ref = O.rmsnorm(x, nw, eps)
    assert np.allclose(xn.cpu().numpy(), xn_ref, rtol=2e-6, atol=0)
    # the fused result against the double dot of the oracle's normalized row
    ry, mag, wn2 = O.matvec(t, Wb, rows, cols, xn_ref)
    err_ref, err_ns = matvec_errors(y1[:rows].cpu().numpy(), ry, mag, wn2, xn_ref, rows, cols, 1)
    print(f"  matvec_rmsnorm {O.TYPE_NAMES[t]:7s} {rows:5d} x {cols:5d}: bit-identical; err {err_ref:.2e} north-star {err_ns:.2e}")
    assert err_ns <= TOL_NORTH_STAR and err_ref <= tol_ref(t, cols)


def test_rmsnorm_rows_strides_no_weight_and_alias(dev):
    rows, dim, ins, outs = 5, 1000, 1024, 1100
    X = O.randn(rows * ins, 9, 2.0)
    Xd = up(X)
    Y = torch.full((rows * outs,), 7.0, dtype=torch.float32, device=dev)
    e = q.Enc()
    arch.encode_rmsnorm(e, q.Buffer.of(Xd), None, q.Buffer.of(Y), rows, dim, 1e-6, ins, outs)
    e.wait()
    got = Y.cpu().numpy().reshape(rows, outs)
    for r in range(rows):
        assert np.allclose(got[r, :dim], O.rmsnorm(X[r * ins:r * ins + dim], None, 1e-6), rtol=2e-6, atol=0)
        assert (got[r, dim:] == 7.0).all()
    w = up(O.randn(dim, 10))
    arch.encode_rmsnorm(e, q.Buffer.of(Xd), q.Buffer.of(w), q.Buffer.of(Xd), rows, dim, 1e-6, ins, ins)  # in place
    e.wait()
    got = Xd.cpu().numpy().reshape(rows, ins)
    for r in range(rows):
        assert np.allclose(got[r, :dim], O.rmsnorm(X[r * ins:r * ins + dim], w.cpu().numpy(), 1e-6), rtol=2e-6, atol=1e-30)
        assert np.array_equal(got[r, dim:], X.reshape(rows, ins)[r, dim:])


def test_matvec_rmsnorm_misuse(dev):
    W = q.Buffer.of(torch.zeros(1 << 22, dtype=torch.uint8, device=dev))
    v = q.Buffer.of(torch.zeros(1 << 16, dtype=torch.float32, device=dev))
    e = q.Enc()
    # codebook formats have no fused norm (src/kernels/quant.mm:110)
    with pytest.raises(q.QuantError, match=r"macseek quant: matvec_rmsnorm unsupported \(type IQ1_S rows 64 cols 2048\)"):
        q.encode_matvec_rmsnorm(e, q.QType.IQ1_S, W, 64, 2048, v, v, 1e-6, v)
    with pytest.raises(q.QuantError, match="matvec_rmsnorm unsupported"):
        q.encode_matvec_rmsnorm(e, q.QType.Q6_K, W, 64, 1000, v, v, 1e-6, v)
    with pytest.raises(q.QuantError, match="matvec_rmsnorm unsupported"):  # wider than the LDS row
        q.encode_matvec_rmsnorm(e, q.QType.Q8_0, W, 16, 16384, v, v, 1e-6, v)


@pytest.mark.parametrize("dim", [1, 255, 1024, 1025, 2048, 3000, 4097, 5120, 6145, 8192, 8193])
def test_rmsnorm_row_lengths(dev, dim):
    """Every number of elements per thread, at its longest row and one past it; rows longer than the registers hold."""
    X, w = O.randn(3 * dim, 20 + dim, 2.0), O.randn(dim, 21)
    Xd, wd = up(X), up(w)
    Y = torch.full((3 * dim + 8,), 7.0, dtype=torch.float32, device=dev)
    e = q.Enc()
    arch.encode_rmsnorm(e, q.Buffer.of(Xd), q.Buffer.of(wd), q.Buffer.of(Y), 3, dim, 1e-6)
    e.wait()
    got = Y.cpu().numpy()
    assert (got[3 * dim:] == 7.0).all()
    for r in range(3):
        assert np.allclose(got[r * dim:(r + 1) * dim], O.rmsnorm(X[r * dim:(r + 1) * dim], w, 1e-6), rtol=2e-6, atol=0)


@pytest.mark.parametrize("t,rows,cols", [(O.Q5_K, 512, 7168), (O.Q6_K, 2048, 5120), (O.IQ4_NL, 33, 12288), (O.BF16, 600, 256)], ids=lambda v: None)
def test_fused_norm_takes_rows_off_16_byte_boundaries(dev, t, rows, cols):
    """Input row and norm weights 4 bytes past a boundary give the bits of aligned ones."""
    arena, (W,) = place_in_arena([O.random_blocks(t, rows * cols, 31, 0.03)])
    x, nw = O.randn(cols, 32, 3.0), (1.0 + 0.2 * O.randn(cols, 33)).astype(np.float32)
    y = []
    for off in (0, 1):
        xd, nwd = (up(np.concatenate([np.zeros(off, np.float32), v])) for v in (x, nw))
        o = torch.zeros(rows, dtype=torch.float32, device=dev)
        e = q.Enc()
        q.encode_matvec_rmsnorm(e, t, W, rows, cols, q.Buffer.of(xd[off:]), q.Buffer.of(nwd[off:]), 1e-6, q.Buffer.of(o))
        e.wait()
        y.append(o)
    assert torch.equal(y[0], y[1]) and bool(y[0].any())


# both prologues of the fused norm on either side of each line between them: block formats in mv_kernel (2560 columns; one
# and several workgroups per CU up to 4096) and mv_tok_kernel (4608 columns; 40 MB; Q8_0 3072 columns, 16 and 30 MB), dense
# types in mv_kernel (2304 columns; thirteen waves a row, one and several workgroups per CU) and mv_tok_kernel (1024 and 2304
# columns; 32 MB); a single row, and rows that leave waves idle
LINES = [
    (O.Q6_K, 301, 2304), (O.Q6_K, 301, 2560), (O.IQ4_NL, 1023, 4096), (O.IQ4_NL, 1029, 4096), (O.Q8_0, 1029, 2816), (O.Q8_0, 1029, 3072),
    (O.Q5_K, 1, 4352), (O.Q5_K, 2049, 4352), (O.Q5_K, 2049, 4608), (O.Q8_0, 2100, 2816), (O.Q8_0, 2100, 3072), (O.Q8_0, 6600, 2304),
    (O.Q8_0, 13801, 2048), (O.Q6_K, 16385, 2816), (O.Q6_K, 17401, 2816), (O.BF16, 1, 2048), (O.BF16, 257, 2304), (O.F32, 33, 512),
    (O.F32, 512, 6144), (O.F32, 513, 6656), (O.F32, 250, 6656), (O.F16, 2050, 1024), (O.F16, 2050, 1280), (O.F16, 2050, 2048),
    (O.F16, 2050, 2304), (O.BF16, 8200, 2048), (O.BF16, 7801, 2048),
]


@pytest.mark.parametrize("t,rows,cols", LINES, ids=lambda v: None)
def test_both_prologues_of_the_fused_norm(dev, t, rows, cols):
    test_fused_equals_norm_then_matvec_and_oracle(dev, t, rows, cols)


# weight rows through LDS, two rows as one, a second workgroup per CU under a fused norm: Q6_K of 17 MB (rows in pairs; an odd
# number of rows; whole waves), 48 and 200 MB (its lines: test_rows_through_lds_by_waves), Q8_0 on either side of 20 MB (pairs) and 40 MB, two
# workgroups from 48 MB (Q5_K with either prologue) and 8 MB (dense; F32 of one and two units a lane)
LARGE = [
    (O.Q6_K, 4000, 5120), (O.Q6_K, 4096, 5120), (O.Q6_K, 4097, 5120), (O.Q6_K, 10300, 2048), (O.Q6_K, 16390, 3584), (O.Q6_K, 119500, 2048),
    (O.Q8_0, 7300, 2560), (O.Q8_0, 7400, 2560), (O.Q8_0, 14800, 2560), (O.Q8_0, 9200, 4096), (O.Q5_K, 16400, 4608), (O.Q5_K, 34200, 2048),
    (O.IQ4_NL, 16800, 5120), (O.F32, 600, 4096), (O.F32, 600, 5120), (O.BF16, 4100, 1280),
]


@pytest.mark.parametrize("t,rows,cols", LARGE, ids=lambda v: None)
def test_fused_norm_of_large_matrices(dev, t, rows, cols):
    test_fused_equals_norm_then_matvec_and_oracle(dev, t, rows, cols)


# Q8_0 rows of 40 MB matrices, which go through LDS where a workgroup's buffers find room beside its activations: the longest
# row that leaves it, one block more, and the longest that a workgroup takes (with the norm and, to compare, without)
@pytest.mark.parametrize("rows,cols", [(2700, 14336), (2720, 14368), (2400, 16384)], ids=lambda v: None)
def test_large_matrices_of_long_rows(dev, rows, cols):
    test_fused_equals_norm_then_matvec_and_oracle(dev, O.Q8_0, rows, cols)


# Q6_K rows through LDS under a fused norm, on either side of each line: six waves a CU and 17 MB (short rows: 2048 columns) or 26
# MB (6144); five waves a CU (4608, 10240 columns), and ten once a second workgroup fits (4608 columns, 48 MB); an odd number of rows
@pytest.mark.parametrize("rows,cols", [(10100, 2048), (10140, 2048), (5150, 6144), (5170, 6144), (7200, 4608), (12690, 4608), (12710, 4608), (11701, 5120), (3572, 10240), (5730, 10240)],
                         ids=lambda v: None)
def test_rows_through_lds_by_waves(dev, rows, cols):
    test_fused_equals_norm_then_matvec_and_oracle(dev, O.Q6_K, rows, cols)
