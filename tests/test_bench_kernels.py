"""The kernels that bench.py names are kernels of the library as it was last built here, and the HBM traffic that it quotes was
counted for them: a kernel that is renamed or gets another template argument does not inherit the figures of the one before."""
import ctypes as C
import json
import os
import re

import pytest

import bench

REPORT = os.path.join(os.path.dirname(__file__), "..", "macseek_amd", "libmsq.kernels.json")
NAMED = (bench.DECODE_GATE_UP, bench.DECODE_DOWN) + bench.PREFILL_GATE_UP + bench.PREFILL_DOWN + bench.MATMUL_CONVERT + (bench.MATVEC_N, bench.ROUTER)


def demangled(name):
    cxx, libc = C.CDLL("libstdc++.so.6"), C.CDLL(None)
    cxx.__cxa_demangle.restype, cxx.__cxa_demangle.argtypes = C.c_void_p, [C.c_char_p, C.c_void_p, C.c_void_p, C.POINTER(C.c_int)]
    libc.free.argtypes = [C.c_void_p]
    status = C.c_int()
    p = cxx.__cxa_demangle(name.encode(), None, None, C.byref(status))
    assert status.value == 0, name
    text = C.cast(p, C.c_char_p).value.decode()
    libc.free(p)
    return re.sub(r"^void ", "", text.replace("(anonymous namespace)::", "").replace("msq::", "")).split("(")[0]


def test_named_kernels_are_in_the_library():
    if not os.path.exists(REPORT):
        pytest.skip("no build report beside the library (built elsewhere)")
    with open(REPORT) as f:
        have = {demangled(k) for ks in json.load(f).values() for k in ks}
    assert not [k for k in NAMED if k not in have]


@pytest.mark.parametrize("name", sorted(bench.TRAFFIC))
def test_traffic_was_counted_for_the_named_kernels(name):
    assert bench.profile_traffic(name)
