"""GPU: the chunked fp32 kernels of wkv5 and wkv5a (head size 64) against the fp64 oracle, where they can go wrong: sequences of
one token, of whole chunks (16 tokens), of whole segments between saved states (48 and 32 tokens) and one off, and decays of
every strength: up to the limit of the chunks' powers ("fast": the tiles with a reference per half chunk) and beyond it ("strong":
half of the channels, so that nearly every head runs step by step).

Tolerance: the fp32 ops' bar of 1e-5, relative to the largest element and to the RMS.  A sum of n fp32 products carries about
sqrt(n) 6e-8; n is at most a few hundred here, and each product has up to six rounded factors: 2e-6.  wkv5a's slow decays
act over the whole sequence (T = 200: 200 x 6e-8)."""
import pytest
import torch

from oracle import err_ratio, max_rel_to_peak
from oracle import wkv5a as A
from oracle import wkv56 as O
from rwkv_cuda_amd import options, wkv5, wkv5a
from _gpu_util import DEV

pytestmark = pytest.mark.gpu
TS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 81, 95, 96, 97, 143, 144, 145, 200]


def _check(names, ref, got):
    for name, a, g in zip(names, ref, got):
        if a is None or float(a.abs().max()) == 0.0:        # the decay gradient when T < 3
            assert float(g.abs().max()) == 0.0, name
            continue
        g = g.detach().double().cpu().reshape(a.shape)
        e, m = err_ratio(a, g), max_rel_to_peak(a, g)
        print(f"  {name}: rms {e:.2e} max {m:.2e}", flush=True)
        assert e <= 1e-5 and m <= 1e-5, name


def _inputs(B, T, H, seed, decays):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s, lo=-1.0, hi=1.0: torch.rand(*s, generator=g) * (hi - lo) + lo
    lo, hi = {"usual": (-1.0, 1.0), "slow": (-8.0, 1.0), "fast": (1.0, 2.83), "strong": (1.0, 3.5)}[decays]      # exp(-exp(3.5)) = 4e-15 a step
    C = H * 64
    return [rnd(B, T, C) for _ in range(3)], [rnd(H, 64, lo=lo, hi=hi), rnd(H, 64), rnd(H, 64, lo=lo, hi=hi), rnd(H, 64)], rnd(B, T, C)


@pytest.mark.parametrize("decays", ["usual", "fast", "strong"])
@pytest.mark.parametrize("T", TS)
def test_wkv5(lib, T, decays):
    B, H = 2, 3
    C = H * 64
    print(f"\nwkv5 fp32 T={T} {decays}", flush=True)
    (r, k, v), (w, u, _, _), gy = _inputs(B, T, H, 7 * T, decays)
    w, u = w.view(C), u.view(C)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u)]
    y = wkv5.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    _check(["y", "gr", "gk", "gv", "gw", "gu"], ref, [y] + [x.grad for x in t])
    with torch.no_grad():                                   # a forward that saves no states
        assert torch.equal(wkv5.RUN_CUDA(B, T, C, H, *t), y)


@pytest.mark.parametrize("decays", ["usual", "slow", "fast", "strong"])
@pytest.mark.parametrize("T", TS)
def test_wkv5a(lib, T, decays):
    B, H = 2, 2
    C = H * 64
    print(f"\nwkv5a T={T} {decays}", flush=True)
    (r, k, v), par, gy = _inputs(B, T, H, 11 * T, decays)
    ref = A.grads(B, T, C, H, r, k, v, *par, gy)
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, *par)]
    y = wkv5a.CUDA_1(*t)
    y.backward(gy.to(DEV))
    _check(["y", "gr", "gk", "gv", "gw1", "gu1", "gw2", "gu2"], ref, [y] + [x.grad for x in t])


def test_one_fast_channel_among_slow_ones(lib):
    """A head takes the references of the fast case, or the steps, as a whole: its ordinary channels must not suffer."""
    B, T, H = 1, 70, 2
    C = H * 64
    (r, k, v), (w, u, _, _), gy = _inputs(B, T, H, 5, "usual")
    w[0, 5], w[0, 40] = 2.5, 6.0
    w, u = w.view(C), u.view(C)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u)]
    y = wkv5.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    _check(["y", "gr", "gk", "gv", "gw", "gu"], ref, [y] + [x.grad for x in t])


def test_sweeps_option_still_runs_the_sequential_kernels(lib):
    B, T, H = 2, 50, 2
    C = H * 64
    (r, k, v), (w, u, _, _), gy = _inputs(B, T, H, 3, "usual")
    w, u = w.view(C), u.view(C)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u)]
    with options.algorithm("sweeps"):
        y = wkv5.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    _check(["y", "gr", "gk", "gv", "gw", "gu"], ref, [y] + [x.grad for x in t])
