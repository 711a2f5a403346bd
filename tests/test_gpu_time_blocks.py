"""GPU: few sequences, cut into blocks of time that run side by side (B H small enough, some 300 tokens at least), against the fp64
oracle where a cut can go wrong: a last block of one token, of one chunk, of one segment between saved states and one off, blocks of
two segments and of more, and many blocks.

Tolerance, fp32: 1e-5 relative to the largest element and to the RMS, the bar of these operators' other tests; a block's state is a sum
in another order, of the same products."""
import pytest
import torch

from oracle import err_ratio, max_rel_to_peak
from oracle import wkv5a as A
from oracle import wkv56 as O
from rwkv_cuda_amd import wkv5, wkv5a
from rwkv_cuda_amd._call import call
from _gpu_util import DEV, garbage

pytestmark = pytest.mark.gpu


def _check(names, ref, got):
    for name, a, g in zip(names, ref, got):
        g = g.detach().double().cpu().reshape(a.shape)
        e, m = err_ratio(a, g), max_rel_to_peak(a, g)
        print(f"  {name}: rms {e:.2e} max {m:.2e}", flush=True)
        assert e <= 1e-5 and m <= 1e-5, name


def _f32_inputs(B, T, H, seed, lo=-1.0, hi=1.0):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s, lo=-1.0, hi=1.0: torch.rand(*s, generator=g) * (hi - lo) + lo
    return [rnd(B, T, H * 64) for _ in range(3)], [rnd(H, 64, lo=lo, hi=hi), rnd(H, 64), rnd(H, 64, lo=lo, hi=hi), rnd(H, 64)], rnd(B, T, H * 64)


@pytest.mark.parametrize("B,H,T", [(1, 3, 257), (1, 3, 288), (2, 2, 289), (1, 3, 337), (1, 1, 1040), (2, 20, 479)])
@pytest.mark.parametrize("decays", [(-8.0, 1.0), (1.0, 2.83), (1.0, 3.5)])             # slow; a reference per half chunk; most heads step by step
@pytest.mark.parametrize("two", [False, True])
def test_fp32(lib, two, decays, B, H, T):
    C = H * 64
    ws = (lib.rwkv_wkv5as_forward_workspace_bytes if two else lib.rwkv_wkv5f32s_forward_workspace_bytes)(B, T, C, H)
    assert ws > 0, "not in blocks"
    print(f"\nwkv5{'a' if two else ''} B={B} H={H} T={T} {decays}", flush=True)
    (r, k, v), par, gy = _f32_inputs(B, T, H, 3 * T + H, *decays)
    if two:
        ref = A.grads(B, T, C, H, r, k, v, *par, gy)
        t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, *par)]
        y = wkv5a.CUDA_1(*t)
    else:
        par = [x.view(C) for x in par[:2]]
        ref = O.wkv5_grads(B, T, C, H, r, k, v, *par, gy)
        t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, *par)]
        y = wkv5.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    _check(["y", "gr", "gk", "gv", "gw1", "gu1", "gw2", "gu2"], ref, [y] + [x.grad for x in t])


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_fp32_inputs_that_are_not_finite_are_the_step_kernels(lib, bad):
    """A head with such an input anywhere gives the bits that it gives without a workspace, where the head runs step by step as a whole;
    the other heads' results, and those of the next call with the same workspace, are as if it were not there."""
    B, H, T = 1, 3, 400
    C = H * 64
    (r, k, v), (w, u, _, _), gy = [[x.to(DEV) for x in y] if isinstance(y, list) else y.to(DEV) for y in _f32_inputs(B, T, H, 9)]
    n = lib.rwkv_wkv5f32s_forward_workspace_bytes(B, T, C, H)
    ws = garbage((n,), torch.uint8)
    whole, blocks, clean = (garbage((B, T, C), torch.float32) for _ in range(3))
    run = lambda r, y: call("rwkv_wkv5f32s_forward_ws", y.device, B, T, C, H, r, k, v, w, u, y, None, 0, ws, n)
    x = r.clone()
    x[0, 390, 64 + 7] = bad
    call("rwkv_wkv5f32s_forward", whole.device, B, T, C, H, x, k, v, w, u, whole, None, 0)
    run(x, blocks)
    run(r, clean)
    assert torch.equal(whole[..., 64:128].nan_to_num(7.0), blocks[..., 64:128].nan_to_num(7.0))
    assert torch.equal(blocks[..., :64], clean[..., :64]) and torch.equal(blocks[..., 128:], clean[..., 128:])
    assert bool(torch.isfinite(blocks[0, :390]).all()) and not bool(torch.isfinite(blocks[0, 390, 64:128]).all()) and bool(torch.isfinite(clean).all())
    # and backwards: the gradients of the other heads are untouched, those of this one are the step kernels'
    t = [z.clone().requires_grad_(True) for z in (r, k, v, w.view(C), u.view(C))]
    good = torch.autograd.grad(wkv5.RUN_CUDA(B, T, C, H, *t), t, gy)
    with torch.no_grad():
        t[0][0, 390, 64 + 7] = bad
    got = torch.autograd.grad(wkv5.RUN_CUDA(B, T, C, H, *t), t, gy)
    for a, b in zip(good, got):
        for h in (0, 2):
            assert torch.equal(a[..., 64 * h:64 * h + 64], b[..., 64 * h:64 * h + 64])
    assert bool(torch.isfinite(got[2][0, 391:]).all()) and bool(torch.isfinite(got[4].view(H, 64)[0]).all())
