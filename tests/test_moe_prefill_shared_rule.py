"""Which prefill MoE calls take a K-quant / Q8_0 shared expert through the few-token kernel: both sides of the lines (112 tokens; 94 experts
in use, or none of more than 48 entries)."""
import ctypes as C

from macseek_amd import _lib


def test_lines():
    few = C.CDLL(_lib.SO).msq_test_prefill_shared_few  # (tokens, experts in use, one of more than 48 entries)
    got = {a: few(*a) for a in [(2, 0, 0), (48, 9, 0), (112, 64, 0), (113, 64, 0), (49, 12, 1), (64, 93, 1), (64, 94, 1), (112, 242, 1), (113, 242, 1)]}
    assert got == {(2, 0, 0): 1, (48, 9, 0): 1, (112, 64, 0): 1, (113, 64, 0): 0, (49, 12, 1): 0, (64, 93, 1): 0, (64, 94, 1): 1, (112, 242, 1): 1,
                   (113, 242, 1): 0}
