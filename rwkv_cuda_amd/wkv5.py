"""RWKV-5 WKV, fp32: drop-in for wkv5/run.py:469-507 (class WKV_5, RUN_CUDA)."""

import torch

from . import options
from ._call import ops

HEAD_SIZE = 64          # the size the matrix-core kernels are written for; any size up to MAX_HEAD_SIZE runs
MAX_HEAD_SIZE = 128


class WKV_5(torch.autograd.Function):
    """Same signature as WKV_5, wkv5/run.py:469-504: r,k,v[B,T,C], w,u with C elements ([C] in the
    reference's checks, :519-520), all fp32, w raw; gw and gu come back in the shape of w and u.  algorithm("sweeps")
    runs the sequential kernels behind the reference's own signature, as do head sizes other than 64."""

    @staticmethod
    def apply(B, T, C, H, r, k, v, w, u):
        return ops().wkv5_f32(B, T, C, H, r, k, v, w, u, options.current_flags())


def RUN_CUDA(B, T, C, H, r, k, v, w, u):
    return WKV_5.apply(B, T, C, H, r, k, v, w, u)
