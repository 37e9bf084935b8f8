"""The fused norm whose sums are taken from registers: row lengths on either side of its batches of eight elements a lane (2048
columns each) and of the 8192 that it holds, formats whose rows end inside a batch, workgroups of fewer than four waves, lines of
the rule (2304 and 2560 columns; dense types alone on a CU and not, 3072 for F32, 4096)."""
import pytest

import oracle as O
from test_matvec_rmsnorm_gpu import test_fused_equals_norm_then_matvec_and_oracle as check

CASES = [
    (O.Q6_K, 300, 2304), (O.Q5_K, 40, 4096), (O.Q5_K, 512, 4352), (O.Q6_K, 1000, 6144), (O.Q6_K, 5, 6400), (O.IQ4_NL, 77, 8192),
    (O.IQ4_NL, 77, 8224), (O.IQ4_NL, 512, 2336), (O.Q8_0, 200, 2560), (O.Q8_0, 1100, 10272), (O.Q6_K, 64, 10496), (O.Q5_K, 1, 12288),
    (O.F32, 100, 3072), (O.F32, 900, 3072), (O.F32, 100, 2816), (O.BF16, 100, 2304), (O.BF16, 1200, 4096), (O.F16, 400, 4352),
    (O.BF16, 200, 8448), (O.F16, 1500, 2304),
]


@pytest.mark.gpu
@pytest.mark.parametrize("t,rows,cols", CASES, ids=lambda v: None)
def test_sums_from_registers(dev, t, rows, cols):
    check(dev, t, rows, cols)
