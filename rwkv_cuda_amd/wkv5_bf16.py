"""RWKV-5 WKV, bf16: drop-in for wkv5_bf16/run.py:44-91 (class WKV_5, RUN_CUDA)."""

import torch

from . import options
from ._call import ops

HEAD_SIZE = 64          # the size the matrix-core kernels are written for; any size up to MAX_HEAD_SIZE runs
MAX_HEAD_SIZE = 128


class WKV_5(torch.autograd.Function):
    """Same signature as WKV_5, wkv5_bf16/run.py:44-88: r,k,v[B,T,C], w,u[H,N], all bf16, w raw."""

    @staticmethod
    def apply(B, T, C, H, r, k, v, w, u):
        return ops().wkv5_bf16(B, T, C, H, r, k, v, w, u, options.current_flags())


def RUN_CUDA(B, T, C, H, r, k, v, w, u):
    return WKV_5.apply(B, T, C, H, r, k, v, w, u)
