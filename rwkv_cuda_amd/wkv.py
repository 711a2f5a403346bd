"""RWKV-4 WKV, fp32: drop-in for wkv/run.py:89-120 (class WKV, RUN_CUDA)."""

import torch

from ._call import ops


class WKV(torch.autograd.Function):
    """Same signature as WKV, wkv/run.py:89-117: w,u[C] (w raw), k,v[B,T,C], fp32."""

    @staticmethod
    def apply(B, T, C, w, u, k, v):
        return ops().wkv4(B, T, C, w, u, k, v)


def RUN_CUDA(B, T, C, w, u, k, v):
    return WKV.apply(B, T, C, w.cuda(), u.cuda(), k.cuda(), v.cuda())
