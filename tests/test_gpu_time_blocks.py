"""GPU: few sequences, cut into blocks of time that run side by side (B H small enough, some 300 tokens at least), against the fp64
oracle where a cut can go wrong: a last block of one token, of one chunk, of one segment between saved states and one off, blocks of
two segments and of more, and many blocks.

Tolerances.  wkv5, wkv5a fp32: 1e-5 relative to the largest element and to the RMS, the bar of these operators' other tests; a block's
state is a sum in another order, of the same products.  rwkv7: fp32 results 4e-7 (some four to eight roundings of 2^-24 a result, as
without blocks; a state at a border is one more product over 64 channels), dw 3e-7 a chunk adding up as a random walk, bf16 results the
rounding of the output.  wkv5 bf16: the bar of the other bf16 kernels, no further from fp64 than fp32 arithmetic with rounded outputs."""
import math

import pytest
import torch

from oracle import err_ratio, max_rel_to_peak
from oracle import wkv5a as A
from oracle import wkv56 as O
from rwkv_cuda_amd import rwkv7_fast_fused as R
from rwkv_cuda_amd import synth, wkv5, wkv5_bf16, wkv5a, wkv6_state
from rwkv_cuda_amd._call import call
from _gpu_util import DEV, assert_no_worse, garbage

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
    # and backwards: the gradients of the other heads are untouched (those of this one: the test below)
    t = [z.clone().requires_grad_(True) for z in (r, k, v, w.view(C), u.view(C))]
    good = torch.autograd.grad(wkv5.RUN_CUDA(B, T, C, H, *t), t, gy)
    with torch.no_grad():
        t[0][0, 390, 64 + 7] = bad
    got = torch.autograd.grad(wkv5.RUN_CUDA(B, T, C, H, *t), t, gy)
    for a, b in zip(good, got):
        for h in (0, 2):
            assert torch.equal(a[..., 64 * h:64 * h + 64], b[..., 64 * h:64 * h + 64])
    assert bool(torch.isfinite(got[2][0, 391:]).all()) and bool(torch.isfinite(got[4].view(H, 64)[0]).all())


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("which", ["r", "k", "v", "gy"])
@pytest.mark.parametrize("t", [5, 200, 391])                # in the first, a middle and the last block
@pytest.mark.parametrize("two", [False, True])
def test_fp32_head_with_an_input_that_is_not_finite(lib, two, t, which, bad):
    """wkv5, wkv5a, both directions: whatever block such an input is in, the head's outputs and gradients, those of its parameters among them, are
    the bits of a call without blocks, where the step kernels do the head; the other heads' are those of a call without that input."""
    B, H, T, name = 2, 3, 400, "as" if two else "f32s"
    C = H * 64
    x, par, gy = _f32_inputs(B, T, H, 11 + t)
    par = par if two else [z.view(C) for z in par[:2]]
    clean = [z.to(DEV) for z in (*x, gy)]
    par = [z.to(DEV) for z in par]
    spoilt = [z.clone() for z in clean]
    spoilt[["r", "k", "v", "gy"].index(which)][1, t, 64 + 7] = bad
    size = lambda what: getattr(lib, f"rwkv_wkv5{name}_{what}_bytes")(B, T, C, H)

    def run(ins, blocks):
        r, k, v, gy = ins
        saved, y, gr, gk, gv = garbage((size("saved"),), torch.uint8), *(garbage((B, T, C), torch.float32) for _ in range(4))
        gpar = [garbage((C,), torch.float32) for _ in par]
        n, m = (size("forward_workspace"), size("backward_workspace")) if blocks else (0, 4 * len(par) * B * C)
        assert not blocks or n > 0 and m > 4 * len(par) * B * C, "not in blocks"
        call(f"rwkv_wkv5{name}_forward_ws", y.device, B, T, C, H, r, k, v, *par, y, saved, saved.numel(), garbage((n,), torch.uint8) if n else None, n)
        call(f"rwkv_wkv5{name}_backward", y.device, B, T, C, H, r, k, v, *par, gy, gr, gk, gv, *gpar, saved, saved.numel(), garbage((m,), torch.uint8), m)
        return [z.view(B, T, H, 64) for z in (y, gr, gk, gv)], [z.view(H, 64) for z in gpar]

    (a, pa), (b, pb), (c, pc) = run(spoilt, False), run(spoilt, True), run(clean, True)
    same = lambda p, q: torch.equal(p.nan_to_num(7.0, 8.0, 9.0), q.nan_to_num(7.0, 8.0, 9.0))
    for i, (whole, blocks, good) in enumerate(zip(a, b, c)):
        hit = i > 0 or which != "gy"                        # (gy is none of the forward's inputs: that head is in blocks there)
        assert same(whole[1, :, 1], blocks[1, :, 1]) if hit else torch.equal(good[1, :, 1], blocks[1, :, 1]), i
        assert torch.equal(blocks[0], good[0]) and torch.equal(blocks[1, :, [0, 2]], good[1, :, [0, 2]]), i
    assert not all(bool(z[1, :, 1].isfinite().all()) for z in b)
    # the parameters' gradients: head 1's of batch row 1 from the step kernels in either call, of row 0 from blocks in one of them
    for i, (whole, blocks, good) in enumerate(zip(pa, pb, pc)):
        assert torch.equal(blocks[[0, 2]], good[[0, 2]]), i
        assert torch.equal(whole[1].isfinite(), blocks[1].isfinite()), i
        ok = whole[1].isfinite()
        assert float((whole[1][ok] - blocks[1][ok]).abs().max() if bool(ok.any()) else 0.0) <= 1e-5 * float(good[1].abs().max()) + 1e-5 * float(whole[1][ok].abs().max() if bool(ok.any()) else 0.0), i


def _f32_backward(lib, two, B, T, H, at):
    """Both directions of wkv5 or wkv5a by the C entry points; at(bytes of the rows, bytes of everything) -> (address, bytes) of the backward's workspace."""
    C, name = H * 64, "as" if two else "f32s"
    (r, k, v), par, gy = _f32_inputs(B, T, H, 17 + T)
    par = par if two else [x.view(C) for x in par[:2]]
    ref = (A.grads if two else O.wkv5_grads)(B, T, C, H, r, k, v, *par, gy)
    r, k, v, gy, *par = (x.to(DEV) for x in (r, k, v, gy, *par))
    n = getattr(lib, f"rwkv_wkv5{name}_saved_bytes")(B, T, C, H)
    saved, y, gr, gk, gv = garbage((n,), torch.uint8), *(garbage((B, T, C), torch.float32) for _ in range(4))
    gpar = [garbage((C,), torch.float32) for _ in par]
    call(f"rwkv_wkv5{name}_forward", y.device, B, T, C, H, r, k, v, *par, y, saved, n)
    address, m = at(4 * len(par) * B * C, getattr(lib, f"rwkv_wkv5{name}_backward_workspace_bytes")(B, T, C, H))
    call(f"rwkv_wkv5{name}_backward", y.device, B, T, C, H, r, k, v, *par, gy, gr, gk, gv, *gpar, saved, n, address, m)
    _check(["y", "gr", "gk", "gv", "gw1", "gu1", "gw2", "gu2"], ref, [y, gr, gk, gv, *gpar])


@pytest.mark.parametrize("two", [False, True])
def test_fp32_backward_with_a_workspace_for_the_rows_only(lib, two):
    """What the backward took before there were blocks of time: whole sequences are walked through, and nothing behind the rows is written."""
    buffer = torch.full((1 << 16,), 7.5, device=DEV)

    def at(rows, everything):
        assert rows < everything and rows % 4 == 0, "not in blocks"
        at.rows = rows
        return buffer.data_ptr(), rows

    _f32_backward(lib, two, 2, 400, 2, at)
    assert bool((buffer[at.rows // 4:] == 7.5).all())


@pytest.mark.parametrize("two", [False, True])
def test_fp32_backward_with_a_workspace_at_any_float(lib, two):
    """The blocks' states are stored and loaded 16 bytes at a time, the rows as single floats: a workspace of any alignment is taken as it
    was before there were blocks, for whole sequences (nothing behind the rows is written)."""
    buffer = torch.full((1 << 18,), 7.5, device=DEV)

    def at(rows, everything):
        assert rows < everything <= 4 * buffer.numel() - 4, "not in blocks"
        at.rows = rows
        return buffer.data_ptr() + 4, everything

    _f32_backward(lib, two, 2, 400, 2, at)
    assert float(buffer[0]) == 7.5 and bool((buffer[1 + at.rows // 4:] == 7.5).all())


def _rwkv7(B, T, H, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=g)
    kk = torch.nn.functional.normalize(n(B, T, H, 64), dim=-1)
    x = [n(B, T, H, 64) * 0.5, n(B, T, H, 64) + 0.5, n(B, T, H, 64) * 0.5, n(B, T, H, 64) * 0.5, -kk, kk * torch.sigmoid(n(B, T, H, 64))]
    return n(B, H, 64, 64) * 0.1, [t.to(dtype).view(B, T, H * 64) for t in x], n(B, T, H * 64).to(dtype), n(B, H, 64, 64) * 0.1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("variant", ["passing", "state", "none"])
@pytest.mark.parametrize("B,T,H", [(1, 256, 2), (2, 272, 1), (1, 33 * 16, 3), (1, 19 * 16, 70)])      # (the last: nothing cut in the forward)
def test_rwkv7(lib, variant, dtype, B, T, H):
    assert lib.rwkv7_workspace_bytes(B, T, H, 1) > 0, "not in blocks"
    print(f"\nrwkv7 {variant} B={B} T={T} H={H} {dtype}", flush=True)
    s0, x, dy, dsT = _rwkv7(B, T, H, dtype, 5 * T + H)
    ins = ([] if variant == "none" else [s0]) + x
    dev = [t.to(DEV).requires_grad_(True) for t in ins]
    op = {"passing": R.RWKV7_STATE_PASSING_CLAMPW_CUDA, "state": R.RWKV7_STATE_CLAMPW_CUDA, "none": R.RWKV7_CLAMPW_CUDA}[variant]
    out = list(op(*dev)) if variant == "passing" else [op(*dev)]
    up = [dy, dsT] if variant == "passing" else [dy]
    got = [z.detach() for z in out] + list(torch.autograd.grad(out, dev, [z.to(DEV) for z in up]))
    with torch.no_grad():                                   # the forward that keeps nothing is cut in the same way
        again = op(*dev)
    assert torch.equal(again[0] if variant == "passing" else again, got[0])
    p = [t.double().to(DEV).requires_grad_(True) for t in ins]          # (the step form in 64 bits, on the GPU for its speed)
    S = p[0] if variant != "none" else torch.zeros(B, H, 64, 64, dtype=torch.float64, device=DEV)
    r, w, k, v, a, b = (t.view(B, T, H, 64) for t in p[-6:])
    d, ys = torch.exp(-math.exp(-0.5) * torch.sigmoid(w)), []
    for t in range(T):
        sa = (S * a[:, t, :, None, :]).sum(-1)
        S = S * d[:, t, :, None, :] + sa[..., None] * b[:, t, :, None, :] + v[:, t, :, :, None] * k[:, t, :, None, :]
        ys.append((S * r[:, t, :, None, :]).sum(-1))
    outs = [torch.stack(ys, 1).view(B, T, H * 64)] + ([S] if variant == "passing" else [])
    want = [z.detach() for z in outs] + list(torch.autograd.grad(outs, p, [z.double().to(DEV) for z in up]))
    names = ["y"] + (["sT"] if variant == "passing" else []) + (["ds0"] if variant != "none" else []) + ["dr", "dw", "dk", "dv", "da", "db"]
    for name, e, g in zip(names, want, got):
        q = float((g.double().view_as(e) - e).norm() / e.norm())
        print(f"  {name}: {q:.2e}", flush=True)
        assert q <= (2.0 ** -8 if g.dtype == torch.bfloat16 else 6e-7 * (T / 16) ** 0.5 if name == "dw" else 4e-7), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,T,forward,backward", [(1, 257, 768, 1, 1), (4, 68, 768, 16, 16), (3, 91, 256, 0, 17), (2, 176, 384, 0, 96), (1, 353, 384, 0, 0),
                                                   (9, 57, 256, 0, 1), (2, 176, 368, 0, 0), (1, 258, 752, 0, 2)])
def test_rwkv7_heads_beyond_a_multiple_of_the_cus(lib, B, H, T, forward, backward, dtype):
    """forward, backward: how many of the last heads are done in blocks there.  The others have the bits of a call without a workspace, these
    differ by the rounding of a state that is summed in another order (one more rounding of 2^-24 a block's product, and a bf16 result may
    fall on the other side)."""
    n = [lib.rwkv7_workspace_bytes(B, T, H, i) for i in (0, 1)]
    assert [m > 0 for m in n] == [forward > 0, backward > 0]
    s0, x, dy, dsT = _rwkv7(B, T, H, dtype, B + H)
    s0, dy, dsT, x = s0.to(DEV), dy.to(DEV), dsT.to(DEV), [t.to(DEV) for t in x]
    f32 = int(dtype == torch.float32)
    new = lambda *s, dt=torch.float32: garbage(s, dt)
    rows = lambda t: t.view(B, T, H, 64).transpose(1, 2).reshape(B * H, -1)
    s, sa = new(B, H, T // 16, 64, 64), new(B, T, H, 64)
    res = []
    for cut in (True, False):                               # (the backward of both from the second one's states)
        # (a workspace that is too small is not used)
        ws = garbage((n[0] if cut else 16 * (B > 1),), torch.uint8)
        y, sT = new(B, T, H * 64, dt=dtype), new(B, H, 64, 64)
        call("rwkv7_forward_ws", y.device, B, T, H, f32, s0, *x, y, sT, s, sa, ws if ws.numel() else None, ws.numel())
        res.append([rows(y), sT.view(B * H, -1), s.view(B * H, -1).clone(), rows(sa).clone()])
    for i, cut in enumerate((True, False)):
        ws = garbage((n[1] if cut else 16 * (B > 1),), torch.uint8)
        ds0, d = new(B, H, 64, 64), [new(B, T, H * 64, dt=dtype) for _ in range(6)]
        call("rwkv7_backward_ws", dy.device, B, T, H, f32, *x, dy, dsT, s, sa, ds0, *d, ws if ws.numel() else None, ws.numel())
        res[i] += [rows(t) for t in d] + [ds0.view(B * H, -1)]
    for z, (got, whole) in enumerate(zip(*res)):
        m = B * H - (forward if z < 4 else backward)
        assert torch.equal(got[:m], whole[:m]), z
        for a, b in zip(got[m:].double(), whole[m:].double()):
            q = float((a - b).norm() / b.norm())
            assert q <= (2.0 ** -8 if got.dtype == torch.bfloat16 else 6e-7 * (T / 16) ** 0.5 if z == 5 else 4e-7), (z, q)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,T", [(1, 257, 768), (1, 3, 1024), (2, 64, 4096)])
def test_rwkv7_states_in_place(lib, B, H, T, dtype):
    """sT in the memory of s0, ds0 in that of dsT: the bits of separate tensors, also where another block of the head writes what one reads."""
    n, f32 = [lib.rwkv7_workspace_bytes(B, T, H, i) for i in (0, 1)], int(dtype == torch.float32)
    assert min(n) > 0
    s0, x, dy, dsT = _rwkv7(B, T, H, dtype, H)
    s0, dy, dsT, x = s0.to(DEV), dy.to(DEV), dsT.to(DEV), [t.to(DEV) for t in x]
    res = []
    for place in (False, True):
        a, b = s0.clone(), dsT.clone()
        sT, ds0 = (a, b) if place else (garbage(a.shape, torch.float32), garbage(b.shape, torch.float32))
        y, s, sa = garbage((B, T, H * 64), dtype), garbage((B, H, T // 16, 64, 64), torch.float32), garbage((B, T, H, 64), torch.float32)
        call("rwkv7_forward_ws", y.device, B, T, H, f32, a, *x, y, sT, s, sa, garbage((n[0],), torch.uint8), n[0])
        d = [garbage((B, T, H * 64), dtype) for _ in range(6)]
        call("rwkv7_backward_ws", y.device, B, T, H, f32, *x, dy, b, s, sa, ds0, *d, garbage((n[1],), torch.uint8), n[1])
        res.append([y, sT, s, sa, ds0] + d)
    same = [torch.equal(g, z) for g, z in zip(*res)]
    assert all(same), same


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("which", ["a", "k"])
def test_rwkv7_heads_that_blocks_cannot_carry_are_done_as_a_whole(lib, which, dtype):
    """A NaN among the inputs, and a transition that overflows over a block where the state itself is zero: the bits of a call without a
    workspace, forward and backward, and other heads are not touched.  (k does not enter the gradient state: the backward of that head
    is not done as a whole, and has no more results that are no number than one that is.)"""
    B, T, H = 1, 512, 3
    s0, x, dy, _ = _rwkv7(B, T, H, dtype, 3)
    head = lambda t, h: t[..., 64 * h:64 * h + 64]
    s0[:, 0] = 0
    head(x[3], 0).zero_()                                   # v
    head(x[4], 0).mul_(-3)                                  # a b^T: a growth of about 4.5 a step
    head(x[5], 0).mul_(3)
    head(dy, 0).zero_()
    head(x[4 if which == "a" else 2], 1)[0, 300, 7] = math.nan
    s0, dy, x = s0.to(DEV), dy.to(DEV), [t.to(DEV) for t in x]
    f32 = int(dtype == torch.float32)
    new = lambda *s, dt=torch.float32: garbage(s, dt)
    res = []
    for cut in (False, True):
        n = [lib.rwkv7_workspace_bytes(B, T, H, i) if cut else 0 for i in (0, 1)]
        ws = [garbage((m,), torch.uint8) if cut else None for m in n]
        y, sT, s, sa, ds0 = new(B, T, H * 64, dt=dtype), new(B, H, 64, 64), new(B, H, T // 16, 64, 64), new(B, T, H, 64), new(B, H, 64, 64)
        d = [new(B, T, H * 64, dt=dtype) for _ in range(6)]
        call("rwkv7_forward_ws", y.device, B, T, H, f32, s0, *x, y, sT, s, sa, ws[0], n[0])
        call("rwkv7_backward_ws", y.device, B, T, H, f32, *x, dy, None, s, sa, ds0, *d, ws[1], n[1])
        res.append([y, *d, sT.transpose(1, 2).reshape(B, 64, H * 64), ds0.transpose(1, 2).reshape(B, 64, H * 64)])
    for z, (whole, blocks) in enumerate(zip(*res)):
        assert torch.equal(head(whole, 0), head(blocks, 0)), z
        if which == "a" or z in (0, 7):
            assert torch.equal(head(whole, 1).nan_to_num(7.0), head(blocks, 1).nan_to_num(7.0)), z
        assert not bool((head(whole, 1).isfinite() & ~head(blocks, 1).isfinite()).any()), z
        assert bool(head(blocks, 2).isfinite().all()) and not torch.equal(head(blocks, 2), garbage((1,), dtype).expand_as(head(blocks, 2)))
    assert bool((head(res[1][0], 0) == 0).all())


@pytest.mark.parametrize("B,H,T", [(1, 2, 321), (1, 1, 384), (2, 1, 385), (1, 3, 449), (1, 9, 700)])
@pytest.mark.parametrize("decays", ["usual", "fast", "mixed"])             # one reference a chunk; up to one per half chunk; some heads step by step
def test_wkv5_bf16_heads_of_128(lib, decays, B, H, T):
    C = H * 128
    assert lib.rwkv_wkv5s_blocks_workspace_bytes(B, T, C, H, 0) > 0 and lib.rwkv_wkv5s_blocks_workspace_bytes(B, T, C, H, 1) > 0, "not in blocks"
    print(f"\nwkv5 N=128 B={B} H={H} T={T} {decays}", flush=True)
    r, k, v, w, u, gy = synth.wkv5_inputs(B, T, C, H, seed=T)
    if decays != "usual":
        lo, hi = {"fast": (-1.0, 2.18), "mixed": (-6.0, 2.3)}[decays]
        w = (torch.rand(w.shape, generator=torch.Generator().manual_seed(5)) * (hi - lo) + lo).to(w.dtype)
    ref = O.wkv5_grads(B, T, C, H, r, k, v, w, u, gy)
    emu = O.emulate_wkv5_bf16(B, T, C, H, r, k, v, w, u, gy)
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u)]
    y = wkv5_bf16.RUN_CUDA(B, T, C, H, *t)
    y.backward(gy.to(DEV))
    with torch.no_grad():                                   # a forward that keeps no states is cut in the same way
        assert torch.equal(wkv5_bf16.RUN_CUDA(B, T, C, H, *t), y)
    for name, a, e, g in zip(["y", "gr", "gk", "gv", "gw", "gu"], ref, emu, [y] + [x.grad for x in t]):
        assert_no_worse(name, a, e.reshape(a.shape), g.reshape(a.shape))


@pytest.mark.parametrize("B,H,T,forward,backward", [(1, 257, 321, 1, 1), (8, 36, 350, 32, 32), (3, 119, 384, 0, 101), (1, 385, 321, 0, 0)])
def test_wkv5_heads_of_128_beyond_a_multiple_of_the_cus(lib, B, H, T, forward, backward):
    """forward, backward: how many of the last heads are done in blocks there.  The others have the bits of a call for whole sequences; these
    differ by the rounding of bf16, 2^-8 at most an element (gw, gu: of each batch row, and again of their sum)."""
    C, WHOLE = H * 128, 0x200
    n = [lib.rwkv_wkv5s_blocks_workspace_bytes(B, T, C, H, i) for i in (0, 1)]
    assert [m > 0 for m in n] == [forward > 0, backward > 0]
    r, k, v, w, u, gy = (x.to(DEV) for x in synth.wkv5_inputs(B, T, C, H, seed=H))
    rows = lambda t: t.view(B, T, H, 128).transpose(1, 2).reshape(B * H, -1)
    ns, nb = lib.rwkv_wkv5s_saved_bytes(B, T, C, H), max(n[1], lib.rwkv_wkv5s_backward_workspace_bytes(B, T, C, H))
    saved, decay, res = garbage((ns,), torch.uint8), garbage((2 * C,), torch.float32), []
    for flags in (0, WHOLE):                                # (the backward of both from the second one's states)
        y, ws = garbage((B, T, C), torch.bfloat16), garbage((n[0],), torch.uint8) if n[0] and not flags else None
        call("rwkv_wkv5s_forward_ws", y.device, B, T, C, H, r, k, v, w, u, y, decay, saved, ns, ws, n[0] if ws is not None else 0, flags)
        res.append([rows(y)])
    for i, flags in enumerate((0, WHOLE)):
        g, gw, gu = [garbage((B, T, C), torch.bfloat16) for _ in range(3)], garbage((H, 128), torch.bfloat16), garbage((H, 128), torch.bfloat16)
        call("rwkv_wkv5s_backward", y.device, B, T, C, H, r, k, v, w, decay, u, gy, *g, gw, gu, saved, ns, garbage((nb,), torch.uint8), nb, flags)
        res[i] += [rows(t) for t in g] + [gw, gu]
    for z, (got, whole) in enumerate(zip(*res)):
        m = (B * H if z < 4 else H) - (forward if z == 0 else backward)
        assert torch.equal(got[:max(m, 0)], whole[:max(m, 0)]), z
        for a, b in zip(got[max(m, 0):].double(), whole[max(m, 0):].double()):
            assert float((a - b).norm() / b.norm()) <= 2.0 ** -8 * (1 if z < 4 else 2), z


@pytest.mark.parametrize("B,H,T,rest", [(1, 257, 321, 1), (8, 36, 350, 32)])
def test_wkv5_heads_of_128_beyond_a_multiple_of_the_cus_keep_what_their_backward_reads(lib, B, H, T, rest):
    """`decay` and `saved` of a forward whose last heads are done in blocks: the bits of whole sequences but for the states of those heads, and the
    gradients from them.  These states differ by roundings of fp32 sums and of bf16 operands, 2^-8 at most; a block's states in the wrong place would be off by their own size."""
    C, WHOLE = H * 128, 0x200
    n = [lib.rwkv_wkv5s_blocks_workspace_bytes(B, T, C, H, i) for i in (0, 1)]
    assert n[0] > 0
    r, k, v, w, u, gy = (x.to(DEV) for x in synth.wkv5_inputs(B, T, C, H, seed=H))
    rows = lambda t: t.view(B, T, H, 128).transpose(1, 2).reshape(B * H, -1)
    ns, nb = lib.rwkv_wkv5s_saved_bytes(B, T, C, H), max(n[1], lib.rwkv_wkv5s_backward_workspace_bytes(B, T, C, H))
    res = []
    for flags in (0, WHOLE):
        y, ws = garbage((B, T, C), torch.bfloat16), garbage((n[0],), torch.uint8) if not flags else None
        saved, decay = garbage((ns // 4,), torch.float32), garbage((2 * C,), torch.float32)
        call("rwkv_wkv5s_forward_ws", y.device, B, T, C, H, r, k, v, w, u, y, decay, saved, ns, ws, n[0] if ws is not None else 0, flags)
        g, gw, gu = [garbage((B, T, C), torch.bfloat16) for _ in range(3)], garbage((H, 128), torch.bfloat16), garbage((H, 128), torch.bfloat16)
        call("rwkv_wkv5s_backward", y.device, B, T, C, H, r, k, v, w, decay, u, gy, *g, gw, gu, saved, ns, garbage((nb,), torch.uint8), nb, flags)
        res.append([decay, saved.view(B * H, -1)] + [rows(t) for t in g] + [gw, gu])
    (decay, saved, *grads), (decay1, saved1, *grads1) = res
    m = B * H - rest
    same = [torch.equal(decay, decay1), torch.equal(saved[:m], saved1[:m])]
    assert all(same), same
    for z, (got, whole) in enumerate(zip([saved[m:]] + grads, [saved1[m:]] + grads1)):
        for a, b in zip(got.double(), whole.double()):
            assert float((a - b).norm() / b.norm()) <= 2.0 ** -8 * (1 if z < 4 else 2), z


@pytest.mark.parametrize("H,T", [(3, 257), (3, 1100), (3, 2300), (64, 1025), (100, 641), (100, 1300)])       # 2, 9, 18 (a scan of its own), 4, 2, 2 blocks of 128 .. 704 tokens
def test_wkv6_state_blocks_of_every_length(lib, H, T):
    """The first pass takes a block's tokens up to 256 at a time, 32 or more a part; three heads of the layer against the oracle."""
    B, C, heads = 1, H * 64, [0, H // 2, H - 1]
    r, k, v, w, u, gy, s0 = synth.wkv6_inputs(B, T, C, H, seed=T + H, state=True)
    t = [x.to(DEV).requires_grad_(True) for x in (r, k, v, w, u, s0)]
    y = wkv6_state.RUN_CUDA(B, T, C, H, *t)
    got = [y] + list(torch.autograd.grad(y, t, gy.to(DEV)))
    some = lambda x: x.reshape(B, T, H, 64)[:, :, heads].reshape(B, T, 3 * 64).contiguous() if x.dim() == 3 and x.shape[1] == T else x.reshape(-1, H, *x.shape[-2:])[:, heads] if x.dim() == 4 else x.reshape(H, 64)[heads]
    a = [some(x) for x in (r, k, v, w, u)]
    s1 = some(s0)
    ref = O.wkv6_grads(B, T, 192, 3, *a, some(gy), s0=s1)
    emu = O.emulate_wkv6_bf16(B, T, 192, 3, *a, some(gy), s0=s1)
    print(f"\nwkv6_state H={H} T={T}", flush=True)
    for name, e, m, g in zip(["y", "gr", "gk", "gv", "gw", "gu", "gs"], ref, emu, got):
        assert_no_worse(name, e, m.reshape(e.shape), some(g.detach()).cpu().reshape(e.shape))
