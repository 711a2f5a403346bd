"""RWKV-6 WKV (no state): drop-in for wkv6/run.py:128-173 (class WKV_6, RUN_CUDA)."""

import torch

from . import options
from ._call import ops

HEAD_SIZE = 64          # the size the matrix-core kernels are written for; any size up to MAX_HEAD_SIZE runs
MAX_HEAD_SIZE = 128


class WKV_6(torch.autograd.Function):
    """Same signature as WKV_6, wkv6/run.py:128-170: r,k,v,w[B,T,C], u[H,N] bf16, w raw.
    The reference wrapper computes ew = -exp(w.float()) (:147) and its kernel applies exp(ew); here the raw
    w goes straight to the kernels, which evaluate the same two exponentials in fp32.
    The fp32-ew entry points rwkv_wkv6_forward/backward stay available for callers of the C ABI."""

    @staticmethod
    def apply(B, T, C, H, r, k, v, w, u):
        return ops().wkv6(B, T, C, H, r, k, v, w, u, options.current_flags())


def RUN_CUDA(B, T, C, H, r, k, v, w, u):
    return WKV_6.apply(B, T, C, H, r, k, v, w, u)
