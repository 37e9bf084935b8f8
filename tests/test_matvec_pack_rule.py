"""How a one-token matvec is launched: rows as one and workgroups per CU on either side of the rule's lines, and the knobs that impose them."""
import ctypes as C
import os
import subprocess
import sys

import oracle as O
from macseek_amd import _lib

CASES = [  # (type, rows, cols, norm): (rows as one, workgroups per CU); 0 rows: another kernel
    ((O.Q6_K, 32768, 1280, 0), (8, 2)), ((O.Q6_K, 32764, 1280, 0), (4, 1)), ((O.Q6_K, 8184, 1280, 0), (4, 1)), ((O.Q6_K, 8192, 1280, 0), (8, 1)),
    ((O.Q6_K, 4096, 5120, 0), (2, 2)), ((O.Q6_K, 3000, 5120, 0), (2, 1)), ((O.Q6_K, 4097, 5120, 0), (1, 1)), ((O.Q6_K, 4096, 5120, 1), (2, 1)),
    ((O.Q5_K, 6144, 2304, 0), (4, 1)), ((O.Q5_K, 3000, 2304, 0), (1, 1)), ((O.Q8_0, 20000, 1280, 0), (8, 1)), ((O.Q8_0, 8192, 1280, 0), (1, 1)),
    ((O.Q8_0, 4096, 5120, 1), (2, 1)), ((O.Q8_0, 2304, 5120, 1), (1, 1)), ((O.BF16, 512, 1280, 0), (0, 0)),
    ((O.Q8_0, 8192, 512, 0), (4, 1)), ((O.Q8_0, 8196, 512, 0), (2, 1)), ((O.Q8_0, 12288, 512, 0), (2, 1)), ((O.Q8_0, 12292, 512, 0), (4, 1)),
    ((O.Q6_K, 8196, 512, 0), (4, 1)), ((O.Q5_K, 7000, 2304, 1), (1, 1)), ((O.Q5_K, 7600, 2304, 1), (4, 1)), ((O.Q5_K, 7000, 2304, 0), (4, 1)),
    ((O.Q6_K, 7000, 2304, 1), (4, 1)),
]


def launch(t, rows, cols, norm):
    per_cu = C.c_int(0)
    return C.CDLL(_lib.SO).msq_test_matvec_pack(t, rows, cols, norm, C.byref(per_cu)), per_cu.value


def test_lines():
    assert [(c, launch(*c)) for c, _ in CASES] == CASES


def test_imposed_workgroups_per_cu_hold_for_packed_rows():
    for wgs in (1, 3):
        code = ("import ctypes as C; L = C.CDLL(%r); p = C.c_int(0)\n"
                "for a in %r: L.msq_test_matvec_pack(*a, C.byref(p)); print(p.value)") % (_lib.SO, [(int(t), r, c, n) for (t, r, c, n), _ in CASES[:6]])
        out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, MSQ_MV_WGS=str(wgs)), check=True, capture_output=True, text=True, timeout=60)
        assert out.stdout.split() == [str(wgs)] * 6
