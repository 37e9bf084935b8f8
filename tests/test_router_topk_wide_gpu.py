"""msq_router_topk on either side of the line between an expert a thread and a wave per token: one to eight waves of experts, the last
token count of the first and the first of the second; fewer than six comparable keys (NaN logits) in the first; and, on the CPU, the lines."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from macseek_amd import _lib, arch, quant as q
from test_router_gpu import test_router_topk_and_route_lists_vs_oracle as check
from util import up



def test_lines():
    # a launch holds fewer than 2^32 threads: many tokens want the form of 64 threads each, whatever the experts
    wide = C.CDLL(_lib.SO).msq_test_router_topk_wide
    got = {a: wide(*a) for a in [(1024, 512), (1025, 512), (1025, 192), (4096, 128), (4097, 128), (1 << 25, 128), (4097, 64), (1 << 25, 64)]}
    assert got == {(1024, 512): 1, (1025, 512): 0, (1025, 192): 0, (4096, 128): 1, (4097, 128): 0, (1 << 25, 128): 0, (4097, 64): 1, (1 << 25, 64): 1}


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_exp", [(1, 64), (3, 512), (37, 384), (1024, 192), (1025, 192), (1030, 128), (1024, 448), (1025, 64), (4096, 128), (4097, 128)], ids=lambda v: None)
def test_both_forms(dev, n, n_exp):
    check(dev, n, n_exp)


@pytest.mark.gpu
def test_nan_logits(dev):
    n, n_exp = 5, 320
    logits = np.full((n, n_exp), np.nan, np.float32)
    logits[1, 7], logits[1, 300] = 1.0, 2.0
    logits[2] = O.randn(n_exp, 3)
    ids, w = torch.full((n, 6), -1, dtype=torch.int32, device=dev), torch.zeros(n, 6, device=dev)
    e = q.Enc()
    arch.encode_router_topk(e, q.Buffer.of(up(logits)), q.Buffer.of(up(np.zeros(n_exp, np.float32))), q.Buffer.of(ids), q.Buffer.of(w), n, n_exp)
    e.wait()
    ids, w = ids.cpu().numpy(), w.cpu().numpy()
    assert (ids[[0, 3, 4]] == 0).all() and (w[[0, 3, 4]] == 0).all()
    assert list(ids[1]) == [300, 7, 0, 0, 0, 0] and (w[1, 2:] == 0).all() and (w[1, :2] > 0).all()
    assert len(set(ids[2])) == 6 and (w[2] > 0).all()
