"""RWKV-6 WKV with initial state: drop-in for wkv6_state/run.py:80-127 (class WKV_6STATE, RUN_CUDA)."""

import torch

from . import options
from ._call import ops

HEAD_SIZE = 64          # the size the matrix-core kernels are written for; any size up to MAX_HEAD_SIZE runs
MAX_HEAD_SIZE = 128


class WKV_6STATE(torch.autograd.Function):
    """Same signature, dtypes and returned gradients as WKV_6STATE, wkv6_state/run.py:80-124:
    r,k,v,w[B,T,C], u[H,N], s[B,H,N,N], all bf16; w is the raw decay parameter."""

    @staticmethod
    def apply(B, T, C, H, r, k, v, w, u, s):
        return ops().wkv6_state(B, T, C, H, r, k, v, w, u, s, options.current_flags())


def RUN_CUDA(B, T, C, H, r, k, v, w, u, s):
    return WKV_6STATE.apply(B, T, C, H, r, k, v, w, u, s)
