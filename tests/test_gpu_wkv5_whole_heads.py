"""GPU: bf16 wkv5 with heads of 128 channels, a workgroup per head (rwkv_wkv5s_*, what wkv5_bf16.RUN_CUDA runs), against the fp64
oracle where it can go wrong: one token, whole chunks (32 tokens) and pairs of them (a saved state each) and one off, and decays
of every strength: slow ones, some beyond what one reference token per chunk carries ("fast": up to the limit of one per half a
chunk), and ones beyond that, whose heads run step by step ("mixed", "strong": nearly all heads).  The bar is that of the other bf16 kernels: no further from fp64 than fp32 arithmetic with rounded outputs."""
import hashlib

import pytest
import torch

from oracle import wkv56 as O
from rwkv_cuda_amd import synth, wkv5_bf16
from _gpu_util import DEV, assert_no_worse

pytestmark = pytest.mark.gpu
N = 128


def _run(B, T, C, H, r, k, v, w, u, gy):
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u)]
    y = wkv5_bf16.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    with torch.no_grad():                                   # a forward that keeps no states
        assert torch.equal(wkv5_bf16.RUN_CUDA(B, T, C, H, *t), y)
    return [y.detach()] + [x.grad for x in t]


def _decays(kind, w):
    if kind == "usual":
        return w
    g = torch.Generator().manual_seed(5)
    lo, hi = {"fast": (-1.0, 2.18), "strong": (1.0, 4.0), "slow": (-8.0, -4.0), "mixed": (-6.0, 3.0)}[kind]      # exp(-exp(4)) = 2e-24 a step
    return (torch.rand(w.shape, generator=g) * (hi - lo) + lo).to(w.dtype)


@pytest.mark.parametrize("decays", ["usual", "slow", "fast", "mixed", "strong"])
@pytest.mark.parametrize("T", [1, 2, 31, 32, 33, 63, 64, 65, 96, 97, 130, 260])
def test_wkv5_whole_heads(lib, T, decays):
    B, H = 2, 2
    C = H * N
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=900 + T)
    w = _decays(decays, w)
    print(f"\nwkv5 N=128 T={T} {decays}", flush=True)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    emu = O.emulate_wkv5_bf16(B, T, C, H, r, k, v, w, u, gy)
    for name, a, e, g in zip(["y", "gr", "gk", "gv", "gw", "gu"], ref, emu, _run(B, T, C, H, r, k, v, w, u, gy)):
        assert_no_worse(name, a, e.reshape(a.shape), g.reshape(a.shape))


def test_one_strong_head_among_others_changes_nothing_else(lib):
    """Every workgroup picks its powers by its own head: the heads without a strong channel give the same bits."""
    B, T, H = 2, 100, 3
    C = H * N
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=31)
    a = _run(B, T, C, H, r, k, v, w, u, gy)
    w = w.clone()
    w.view(H, N)[1, 70] = 2.5
    b = _run(B, T, C, H, r, k, v, w, u, gy)
    for x, y in zip(a[:4], b[:4]):
        x, y = x.view(B, T, H, N), y.view(B, T, H, N)
        assert torch.equal(x[:, :, 0], y[:, :, 0]) and torch.equal(x[:, :, 2], y[:, :, 2]) and not torch.equal(x[:, :, 1], y[:, :, 1])


@pytest.mark.parametrize("decays", ["fast", "mixed", "strong"])
@pytest.mark.parametrize("T", [1, 31, 33, 64, 97, 260])
def test_wkv5_head_size_64_with_a_strong_decay(lib, T, decays):
    """Head size 64 belongs to the one-sweep kernels until one channel of the layer decays too fast for them."""
    B, H = 2, 3
    C = H * 64
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=1200 + T)
    w = _decays(decays, w)
    print(f"\nwkv5 N=64 T={T} {decays}", flush=True)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    emu = O.emulate_wkv5_bf16(B, T, C, H, r, k, v, w, u, gy)
    for name, a, e, g in zip(["y", "gr", "gk", "gv", "gw", "gu"], ref, emu, _run(B, T, C, H, r, k, v, w, u, gy)):
        assert_no_worse(name, a, e.reshape(a.shape), g.reshape(a.shape))


@pytest.mark.parametrize("w1", [1.3125, 1.3203125, 1.5, 2.1875, 2.203125, 2.84375])
@pytest.mark.parametrize("head", [64, 128])
def test_wkv5_around_the_thresholds(lib, head, w1):
    """One channel at the decays where the kernels (one-sweep or whole heads), or the reference tokens, change."""
    B, T, H = 1, 70, 2
    C = H * head
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=77)
    w = w.clamp(max=1.25)
    w.view(-1)[head + 9] = w1
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    emu = O.emulate_wkv5_bf16(B, T, C, H, r, k, v, w, u, gy)
    for name, a, e, g in zip(["y", "gr", "gk", "gv", "gw", "gu"], ref, emu, _run(B, T, C, H, r, k, v, w, u, gy)):
        assert_no_worse(name, a, e.reshape(a.shape), g.reshape(a.shape))


# B, T, heads, head size, range of the raw decays -> the bits of y, gr, gk, gv, gw, gu (heads of 64: layers with a strong decay)
BITS = {
    (2, 300, 16, 128, -1.5, 0.5): "9e5d287c9604 c816c03755cf 9aefa4db7628 bbe91d845816 b423a4898c9d 278fcac95b29",
    (3, 97, 20, 128, -1, 2.18): "287d8d19bd15 28c8d598c883 d8aeacb94e1d feaffe1c6659 36b35110b6e8 5905df063a65",
    (4, 200, 24, 64, -2, 2.18): "bf0a6042268c a01564a7c684 7e1cda288c1c 3031bdeb0626 2e686ef0c88a b31c2582b0ee",
}


@pytest.mark.parametrize("case", BITS, ids=str)
def test_the_order_of_the_sums_is_fixed(lib, case):
    """Whole sequences have given these bits since the kernels were first written, whatever the split of the work among waves: every sum in its
    order, the products of a split pair unrounded before their remainder is taken.  Inputs are multiples of 1/128 from integers, the same
    on every machine."""
    B, T, H, head, lo, hi = case
    g = torch.Generator().manual_seed(T)
    draw = lambda a, b, *s: (torch.randint(int(a * 128), int(b * 128) + 1, s, generator=g) / 128).to(torch.bfloat16)
    C = H * head
    r, k, v, gy = (draw(-1, 1, B, T, C) for _ in range(4))
    got = _run(B, T, C, H, r, k, v, draw(lo, hi, H, head), draw(-0.5, 0.5, H, head), gy)
    digest = lambda x: hashlib.sha256(x.detach().cpu().contiguous().view(torch.uint8).numpy().tobytes()).hexdigest()[:12]
    assert [digest(x) for x in got] == BITS[case].split()
