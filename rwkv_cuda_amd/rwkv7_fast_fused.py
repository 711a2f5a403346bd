"""RWKV-7 clamp-w, bf16 or fp32 (the dtype of r selects the mode the reference fixes at build time with DTYPE /
-D_FP32_, rwkv7_cuda_benchmark.py:14,76,102): drop-ins for
rwkv7_fast_fused/rwkv7_cuda_benchmark_state_passing.py:75-103 (RWKV7_STATE_PASSING_CLAMPW_CUDA_OP, ..._CUDA),
rwkv7_fast_fused/rwkv7_cuda_benchmark_state.py:75-102 (RWKV7_STATE_CLAMPW_CUDA_OP, ..._CUDA: initial state only) and
rwkv7_fast_fused/rwkv7_cuda_benchmark.py:76-100 (RWKV7_CLAMPW_CUDA_OP, ..._CUDA: no state).
The *_OP classes take r..b as [B,T,H,64], the functions as [B,T,H*64]."""

import torch

from . import options
from ._call import ops

HEAD_SIZE = 64
CHUNK_LEN = 16


class RWKV7_STATE_PASSING_CLAMPW_CUDA_OP(torch.autograd.Function):
    """apply(s0, r, w, k, v, a, b) -> (y[B,T,H*N], sT); r..b are [B,T,H,N] bf16 (or all fp32), s0/sT fp32 [B,H,N,N]."""

    @staticmethod
    def apply(s0, r, w, k, v, a, b):
        return ops().rwkv7_passing(s0, r, w, k, v, a, b, options.current_flags(), False)


def RWKV7_STATE_PASSING_CLAMPW_CUDA(s0, r, w, k, v, a, b):
    return ops().rwkv7_passing(s0, r, w, k, v, a, b, options.current_flags(), True)


class RWKV7_STATE_CLAMPW_CUDA_OP(torch.autograd.Function):
    """apply(s0, r, w, k, v, a, b) -> y[B,T,H,N]; backward gives (ds0, dr, dw, dk, dv, da, db)
    (rwkv7_cuda_benchmark_state.py:77-98)."""

    @staticmethod
    def apply(s0, r, w, k, v, a, b):
        return ops().rwkv7_state(s0, r, w, k, v, a, b, 0, False)


def RWKV7_STATE_CLAMPW_CUDA(s0, r, w, k, v, a, b):
    return ops().rwkv7_state(s0, r, w, k, v, a, b, 0, True)


class RWKV7_CLAMPW_CUDA_OP(torch.autograd.Function):
    """apply(r, w, k, v, a, b) -> y[B,T,H,N] from a zero state; backward gives (dr, dw, dk, dv, da, db)
    (rwkv7_cuda_benchmark.py:78-96)."""

    @staticmethod
    def apply(r, w, k, v, a, b):
        return ops().rwkv7(r, w, k, v, a, b, 0, False)


def RWKV7_CLAMPW_CUDA(r, w, k, v, a, b):
    return ops().rwkv7(r, w, k, v, a, b, 0, True)
