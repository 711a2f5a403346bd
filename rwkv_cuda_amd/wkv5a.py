"""RWKV-5 WKV with two-sided decay and bonus, fp32: drop-in for wkv5a/run.py:100-157 (class WKV_5A, CUDA_1)."""

import torch

from . import options
from ._call import ops

HEAD_SIZE = 64           # runs on the chunked matrix-core kernels, other sizes on the row kernels
MAX_HEAD_SIZE = 128


class WKV_5A(torch.autograd.Function):
    """Same signature as WKV_5A, wkv5a/run.py:100-154: r,k,v[B,T,C]; w1,u1,w2,u2[H,N]; all fp32, w raw.
    The reference reads B,T,C,H from module globals (:111-115); here they come from the tensors.
    State element [i][j] (i = value channel) decays by exp(-exp(w1[j])) * exp(-exp(w2[i])), and the
    current token's bonus is u1[j] + u2[i]."""

    @staticmethod
    def apply(r, k, v, w1, u1, w2, u2):
        return ops().wkv5a(r, k, v, w1, u1, w2, u2, options.current_flags())


def CUDA_1(r, k, v, w1, u1, w2, u2):
    return WKV_5A.apply(r, k, v, w1, u1, w2, u2)
