"""GPU: wkv4 at the lengths where the cut of a sequence into segments changes (up to 64, 128, 256, 512 and 1024 steps, blocks of 512 beyond,
with fewer channels a workgroup where at most 128 pieces of channels exist), from both sides and with channels that leave the last
workgroup partly empty, against the fp64 oracle.

Tolerance: a step rounds a state's sums four times by 2^-24, and of T steps they add up like a random walk: sqrt(4 * 1600) 2^-24 = 5e-6,
twice that for the ratio of two such sums."""
import pytest
import torch

from oracle import wkv4 as O4
from oracle import err_ratio, max_rel_to_peak
from rwkv_cuda_amd import synth, wkv
from _gpu_util import DEV

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("B,T,C", [(3, 7, 65), (2, 63, 63), (2, 64, 129), (2, 65, 31), (2, 128, 33), (2, 129, 17), (2, 256, 15), (2, 257, 16), (2, 271, 47),
                                   (9, 496, 5), (1, 512, 33), (2, 513, 9), (129, 33, 1), (65, 64, 65), (129, 65, 1), (65, 128, 33),
                                   (129, 129, 1), (65, 250, 17), (129, 257, 1), (65, 500, 17), (8, 1025, 256), (129, 1025, 1), (43, 1537, 33), (1, 1600, 9)])
def test_segments(lib, B, T, C):
    print(f"\nwkv4 B={B} T={T} C={C}", flush=True)
    w_raw, u, k, v, gy = synth.wkv4_inputs(B, T, C, seed=31)
    ref = O4.grads(B, T, C, w_raw, u, k, v, gy)
    t = [x.to(DEV).requires_grad_(True) for x in (w_raw, u, k, v)]
    y = wkv.WKV.apply(B, T, C, *t)
    y.backward(gy.to(DEV))
    torch.cuda.synchronize()
    for name, a, g in zip(["y", "gw", "gu", "gk", "gv"], ref, [y] + [x.grad for x in t]):
        got = g.detach().cpu()
        assert err_ratio(a, got) <= TOL and max_rel_to_peak(a, got) <= TOL, name
