"""GPU: wkv5 and wkv5a heads with a decay that is too fast for the powers of the chunked kernels, or is no number.  They run step
by step, so the decay that acts is the true one, which shows where nothing else hides it (tokens without a key or value of
their own), and a NaN parameter reaches the outputs and its gradient.

Tolerance: bf16 outputs, the bar of the other bf16 kernels (no further from fp64 than fp32 steps with rounded outputs).  fp32, 1e-5 of an element, not of the largest one: an output here is a handful of products of fp32 factors, with a
decay whose log (at most 90) is rounded to fp32: 90 x 6e-8."""
import pytest
import torch

from oracle import wkv56 as O
from oracle import wkv5a as A
from rwkv_cuda_amd import synth, wkv5, wkv5_bf16, wkv5a
from rwkv_cuda_amd._call import call
from _gpu_util import DEV, assert_no_worse

pytestmark = pytest.mark.gpu


def _f32_inputs(B, T, H, seed):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.rand(*s, generator=g) * 2 - 1
    return [rnd(B, T, H * 64) for _ in range(3)] + [rnd(H, 64) for _ in range(4)] + [rnd(B, T, H * 64)]


def _run_f32(two, r, k, v, w1, u1, w2, u2, gy):
    B, T, C = r.shape
    H = w1.shape[0]
    t = [x.to(DEV).requires_grad_(True) for x in ((r, k, v, w1, u1, w2, u2) if two else (r, k, v, w1.reshape(C), u1.reshape(C)))]
    y = wkv5a.CUDA_1(*t) if two else wkv5.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    return [y.detach().cpu()] + [x.grad.cpu() for x in t]


@pytest.mark.parametrize("two", [False, True])
def test_fp32_fast_decays_act_as_they_are(lib, two):
    B, T, H = 2, 50, 3
    C = H * 64
    r, k, v, w1, u1, w2, u2, gy = _f32_inputs(B, T, H, 11)
    w1[0] = torch.linspace(2.80, 2.84, 64)           # either side of the border
    w1[1, 7], w1[1, 20] = 3.0, 4.5                   # e^-20 and e^-90 a step among ordinary channels
    if two:
        w2[2, 30] = 3.0
    k.view(B, T, H, 64)[:, 17::3] = 0                # pairs of tokens without a key: what is left of the state is all they see
    k.view(B, T, H, 64)[:, 18::3] = 0
    r, k, v, w1, u1, w2, u2, gy = [x.double() for x in (r, k, v, w1, u1, w2, u2, gy)]
    ref = A.grads(B, T, C, H, r, k, v, w1, u1, w2, u2, gy) if two else O.wkv5_grads(B, T, C, H, r, k, v, w1.reshape(C), u1.reshape(C), gy)
    got = _run_f32(two, *[x.float() for x in (r, k, v, w1, u1, w2, u2, gy)])
    for name, a, x in zip(["y", "gr", "gk", "gv", "gw1", "gu1", "gw2", "gu2"], ref, got):
        a, x = a.reshape(x.shape), x.double()
        e = float((a - x).abs().max() / a.abs().max())
        print(f"  {name}: max {e:.1e}", flush=True)
        assert e <= 1e-5, name
    # a head whose channels are all fast and a token without keys: y is e^l times a product, far below the other tokens'
    w1 = torch.full((H, 64), 3.2, dtype=torch.float64)
    w2 = torch.full((H, 64), -30.0, dtype=torch.float64)
    args = (r, k, v, w1, u1, w2, u2)
    ref = A.grads(B, T, C, H, *args, gy) if two else O.wkv5_grads(B, T, C, H, r, k, v, w1.reshape(C), u1.reshape(C), gy)
    got = _run_f32(two, *[x.float() for x in (*args, gy)])
    a, x = ref[0].reshape(B, T, C)[:, 18::3], got[0].double()[:, 18::3]       # two steps behind the last key
    assert 0 < float(a.abs().max()) < 1e-9
    assert float((a - x).abs().max() / a.abs().max()) <= 1e-5


@pytest.mark.parametrize("two", [False, True])
def test_fp32_nan_decay_is_not_swallowed(lib, two):
    B, T, H = 1, 40, 3
    x = _f32_inputs(B, T, H, 12)
    clean = _run_f32(two, *x)
    for i in ([3, 5] if two else [3]):
        x[i] = x[i].clone()
        x[i][1, 9] = float("nan")
        got = _run_f32(two, *x)
        y, c = (z[0].view(B, T, H, 64) for z in (got, clean))
        # a decay of key channel 9 meets every output of the head, one of value channel 9 its own
        hit = y[:, 1:, 1] if i == 3 else y[:, 1:, 1, 9]
        assert torch.isnan(hit).all() and torch.equal(y[:, :, 0], c[:, :, 0]) and torch.equal(y[:, :, 2], c[:, :, 2])
        g = got[4 if i == 3 else 6].view(H, 64)
        assert torch.isnan(g[1, 9]) and torch.isfinite(g[0]).all() and torch.isfinite(g[2]).all()
        x[i] = torch.nan_to_num(x[i])


def _run_bf16(B, T, C, H, r, k, v, w, u, gy):
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u)]
    y = wkv5_bf16.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    with torch.no_grad():
        assert torch.equal(wkv5_bf16.RUN_CUDA(B, T, C, H, *t).view(torch.int16), y.view(torch.int16))
    return [y.detach().cpu()] + [x.grad.cpu() for x in t]


@pytest.mark.parametrize("B,T,H,N", [(2, 50, 3, 64), (1, 300, 2, 64), (2, 50, 3, 128), (1, 100, 2, 128)])
def test_bf16_fast_decays_act_as_they_are(lib, B, T, H, N):
    """(1, 300, 2, 64) runs as blocks of time where no decay is strong."""
    C = H * N
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=60 + T)
    w = w.clone()
    w[0] = 3.0                                       # e^-20 a step
    w[1, 3], w[1, 9] = 2.1875, 1.5                   # the last decay of the chunked kernels
    k = k.clone()
    k.view(B, T, H, N)[:, 17::3] = 0
    k.view(B, T, H, N)[:, 18::3] = 0
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    emu = O.emulate_wkv5_bf16(B, T, C, H, r, k, v, w, u, gy)
    got = _run_bf16(B, T, C, H, r, k, v, w, u, gy)
    for name, a, e, x in zip(["y", "gr", "gk", "gv", "gw", "gu"], ref, emu, got):
        assert_no_worse(name, a, e.reshape(a.shape), x.reshape(a.shape))
    a, e, x = (z.view(B, T, H, N)[:, 18::3, 0] for z in (ref[0], emu[0], got[0]))        # two steps behind the last key
    assert 0 < float(a.abs().max()) < 1e-6
    assert_no_worse("y behind the last key", a / a.abs().max(), e.double() / a.abs().max(), x.double() / a.abs().max())


@pytest.mark.parametrize("B,T,H,N", [(2, 50, 3, 64), (1, 300, 3, 64), (2, 70, 3, 128)])
def test_bf16_nan_decay_is_not_swallowed(lib, B, T, H, N):
    C = H * N
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=90 + T)
    w = w.clone()
    w[0, 5] = 1.5                                    # (head 0: a layer of the whole-head kernels either way)
    clean = _run_bf16(B, T, C, H, r, k, v, w, u, gy)
    w[1, 9] = float("nan")
    got = _run_bf16(B, T, C, H, r, k, v, w, u, gy)
    y, c = (z[0].view(B, T, H, N) for z in (got, clean))
    assert torch.isnan(y[:, 32:, 1]).all() and torch.equal(y[:, :, 0], c[:, :, 0]) and torch.equal(y[:, :, 2], c[:, :, 2])
    gw = got[4].view(H, N)
    assert torch.isnan(gw[1, 9]) and torch.isfinite(gw[0]).all() and torch.isfinite(gw[2]).all()


@pytest.mark.parametrize("B,T,H", [(2, 100, 3), (1, 300, 2)])
def test_bf16_head_that_the_forward_gave_up_is_redone_by_the_backward(lib, B, T, H):
    """A one-sweep forward that gives a head up says so in the head's flag words behind the saved states, and leaves no states worth
    anything: here both are written by hand.  (1, 300, 2) runs as blocks of time."""
    C = H * 64
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=70 + T)
    w = w.clamp(max=1.25)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    emu = O.emulate_wkv5_bf16(B, T, C, H, r, k, v, w, u, gy)
    d = [x.to(DEV) for x in (r, k, v, w, u, gy)]
    bf = dict(device=DEV, dtype=torch.bfloat16)
    y, decay = torch.empty(B, T, C, **bf), torch.empty(2 * C, device=DEV)
    nsv = lib.rwkv_wkv5s_saved_bytes(B, T, C, H)
    saved = torch.empty(nsv, device=DEV, dtype=torch.uint8)
    call("rwkv_wkv5s_forward", DEV, B, T, C, H, *d[:5], y, decay, saved, nsv, 0)
    per_head = (T + 63) // 64 * 64 * 64 * 3
    at = B * H * per_head                                           # the flag words, eight a head
    assert int(saved[at:at + 32 * B * H].max()) == 0
    saved[(B * H - 1) * per_head:at] = 0x41                         # the last head
    saved[at + 32 * (B * H - 1)] = 1
    gr, gk, gv = (torch.empty(B, T, C, **bf) for _ in range(3))
    gw, gu = torch.empty(H, 64, **bf), torch.empty(H, 64, **bf)
    n = lib.rwkv_wkv5s_backward_workspace_bytes(B, T, C, H)
    ws = torch.empty(n, device=DEV, dtype=torch.uint8)
    call("rwkv_wkv5s_backward", DEV, B, T, C, H, d[0], d[1], d[2], d[3], decay, d[4], d[5], gr, gk, gv, gw, gu, saved, nsv, ws, n, 0)
    for name, a, e, x in zip(["y", "gr", "gk", "gv", "gw", "gu"], ref, emu, [y, gr, gk, gv, gw, gu]):
        assert_no_worse(name, a, e.reshape(a.shape), x.reshape(a.shape))


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("two", [False, True])
def test_fp32_elements_that_are_not_finite_stay_where_they_act(lib, two, bad):
    """In the middle of a chunk, one input at a time: the outputs and gradients that meet the element are not finite, all others of
    its head are what they are without it, and other heads keep their bits."""
    B, T, H, h, t0, c0 = 2, 60, 3, 1, 23, 9
    x = _f32_inputs(B, T, H, 13)
    clean = [z.view(-1, T, H, 64) for z in _run_f32(two, *x)[:4]]
    t = torch.arange(T)
    upto, since, at = t <= t0, t >= t0, t == t0
    every, one = torch.ones(64, dtype=torch.bool), torch.arange(64) == c0
    # input -> (tokens, channels) of y, gr, gk, gv that it reaches
    reach = {0: [(at, every), None, (upto, one), (upto, every)], 1: [(since, every), (since, one), None, (at, every)],
             2: [(since, one), (since, every), (at, every), None], 7: [None, (at, every), (upto, every), (upto, one)]}
    for i, hits in reach.items():
        y = list(x)
        y[i] = x[i].clone()
        y[i].view(B, T, H, 64)[1, t0, h, c0] = bad
        got = [z.view(-1, T, H, 64) for z in _run_f32(two, *y)[:4]]
        for name, a, g, hit in zip(("y", "gr", "gk", "gv"), clean, got, hits):
            want = torch.zeros(T, 64, dtype=torch.bool) if hit is None else hit[0][:, None] & hit[1][None, :]
            assert torch.equal(~torch.isfinite(g[1, :, h]), want), (i, name)
            assert float((a[1, :, h] - g[1, :, h])[~want].abs().max() / a.abs().max()) <= 1e-5, (i, name)
            assert torch.equal(a[0], g[0]) and torch.equal(a[1, :, [0, 2]], g[1, :, [0, 2]]), (i, name)
