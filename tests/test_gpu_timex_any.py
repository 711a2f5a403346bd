"""GPU: depthwise_conv1d at the lengths and batch sizes that are not whole tiles (timex_conv_any, timex_gw_any), against the fp64
oracle: one block of steps, a block and a piece, odd numbers of blocks, the longest sequence, batches of one row up to more than
one unit, batch groups that are summed by a second kernel and ones that are not.

Tolerance: the fp32 ops' bar of 1e-5.  An operand keeps 22 bits (a product 2^-21), sums are fp32: n products leave about
sqrt(n) 2^-24 + 2^-21 of their scale, 1e-6 at n = 4096 x 33."""
import pytest
import torch

from oracle import err_ratio, max_rel_to_peak
from oracle import timex as OT
from rwkv_cuda_amd import depthwise_conv1d, synth
from _gpu_util import DEV

pytestmark = pytest.mark.gpu


def _check(B, C, T, w, k, g, eps=0.25):
    out, gw, gk = OT.grads(w, k, g, B, C, T)
    t = [x.to(DEV).requires_grad_(True) for x in (w, k)]
    x = depthwise_conv1d.RUN_CUDA(*t, B, C, T, eps)
    x.backward(g.to(DEV))
    for name, a, got in (("x", out + eps, x), ("gw", gw, t[0].grad), ("gk", gk, t[1].grad)):
        got = got.detach().double().cpu()
        e, m = err_ratio(a, got), max_rel_to_peak(a, got)
        print(f"  {name}: rms {e:.2e} max {m:.2e}", flush=True)
        assert e <= 1e-5 and m <= 1e-5, name


@pytest.mark.parametrize("T", [4, 8, 28, 32, 36, 60, 100, 516, 1000, 1028, 1056, 1500, 2048, 4092, 4096])
@pytest.mark.parametrize("B", [1, 2, 5, 13])
def test_shapes(lib, B, T):
    print(f"\ntimex any B={B} T={T}", flush=True)
    _check(B, 3, T, *synth.timex_inputs(B, 3, T, seed=B + T))


@pytest.mark.parametrize("B,C,T", [(7, 5, 96), (16, 2, 772), (31, 2, 68), (32, 3, 100), (33, 2, 36), (64, 1, 1500), (70, 2, 4), (3, 600, 52)])
def test_more_batches(lib, B, C, T):
    print(f"\ntimex any B={B} C={C} T={T}", flush=True)
    _check(B, C, T, *synth.timex_inputs(B, C, T, seed=B + C + T))


def test_reference_signature_gives_per_batch_kernel_gradients(lib):
    from rwkv_cuda_amd._call import call
    B, C, T = 3, 4, 76
    w, k, g = synth.timex_inputs(B, C, T, seed=9)
    d = [x.to(DEV) for x in (w, k, g)]
    gw, gk = torch.empty(B, C, T, device=DEV), torch.empty(B, C, T, device=DEV)
    call("rwkv_timex_backward", d[0].device, *d, gw, gk, B, C, T)
    ref_gw, ref_gk = OT.grads_closed_form(*(x.double() for x in (w, k, g)), B, C, T)
    assert max_rel_to_peak(ref_gw, gw.double().cpu()) <= 1e-5 and max_rel_to_peak(ref_gk, gk.double().cpu()) <= 1e-5


def test_rows_of_very_different_size(lib):
    """A unit shares one power of two: the small rows of a unit keep their accuracy down to 2^-28 of its largest element."""
    B, C, T = 6, 2, 500
    w, k, g = synth.timex_inputs(B, C, T, seed=4)
    scale = torch.tensor([1.0, 1e-4, 1e3, 1e-2, 1.0, 1e-3]).view(B, 1, 1)
    out, gw, gk = OT.grads(w, k * scale, g * scale, B, C, T)
    t = [x.to(DEV).requires_grad_(True) for x in (w, k * scale)]
    x = depthwise_conv1d.RUN_CUDA(*t, B, C, T, 0.0)
    x.backward((g * scale).to(DEV))
    for b in range(B):
        assert max_rel_to_peak(out[b], x[b].detach().double().cpu()) <= 1e-5 and max_rel_to_peak(gk[b], t[1].grad[b].double().cpu()) <= 1e-5, b
