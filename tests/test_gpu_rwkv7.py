"""GPU parity: rwkv7 clamp-w with state passing through the C ABI against the CPU oracle."""
import math

import pytest
import torch

from oracle import rwkv7 as O
from oracle import err_ratio
from rwkv_cuda_amd import options, synth, rwkv7_fast_fused as R
from rwkv_cuda_amd._call import call
from _gpu_util import DEV, assert_no_worse

pytestmark = pytest.mark.gpu
NAMES = ["y", "sT", "ds0", "dr", "dw", "dk", "dv", "da", "db"]


def _run(args, splits=1):
    s0, r, w, k, v, a, b, dy, dsT = args
    B, T, H, N = r.shape
    t = [x.to(DEV).requires_grad_(True) for x in (s0, r, w, k, v, a, b)]
    S = t[0]
    ys = []
    step = T // splits
    for c in range(splits):
        sl = slice(c * step, (c + 1) * step)
        y, S = R.RWKV7_STATE_PASSING_CLAMPW_CUDA(S, *(x[:, sl].contiguous().view(B, step, H * N) for x in t[1:]))
        ys.append(y)
    y = torch.cat(ys, 1)
    torch.autograd.backward([y, S], [dy.to(DEV).view(B, T, H * N), dsT.to(DEV)])
    torch.cuda.synchronize()
    return [y.detach().view(B, T, H, N), S.detach()] + [x.grad for x in t]


@pytest.mark.parametrize("algo", ["chunked", "sweeps"])
@pytest.mark.parametrize("B,T,H", [(2, 32, 2), (1, 64, 3), (3, 16, 1)])
def test_rwkv7_small(lib, B, T, H, algo):
    """Both kernel families: the chunked matrix-core kernels (default) and the step-by-step recurrence."""
    print(f"\nrwkv7 B={B} T={T} H={H} {algo}", flush=True)
    args = synth.rwkv7_inputs(B, T, H, 64, seed=31)
    ref = O.grads(*args)
    emu = O.emulate_bf16(*args)
    with options.algorithm(algo):
        got = _run(args)
    for name, a, e, g in zip(NAMES, ref, emu, got):
        assert_no_worse(name, a, e, g)


def test_rwkv7_chained_calls_small(lib):
    """Four chained T/4 calls (state handed over) against the fp64 oracle of one T call."""
    B, T, H = 2, 128, 2
    args = synth.rwkv7_inputs(B, T, H, 64, seed=32)
    ref = O.grads(*args)
    emu = O.emulate_bf16(*args)
    got = _run(args, splits=4)
    for name, a, e, g in zip(NAMES, ref, emu, got):
        assert_no_worse(name, a, e, g)


def test_rwkv7_full_size_chain_equals_one_call(lib):
    """B8 T4096 C4096 (H64): 4 x T1024 chained must reproduce one T4096 call.  Forward values are
    bit-identical (same arithmetic, states handed over in fp32); gradients agree to rounding."""
    B, T, H = 8, 4096, 64
    args = synth.rwkv7_inputs(B, T, H, 64, seed=42)
    print("\nrwkv7 full size: one call", flush=True)
    one = _run(args)
    print("rwkv7 full size: four chained calls", flush=True)
    four = _run(args, splits=4)
    assert torch.equal(one[0], four[0]) and torch.equal(one[1], four[1])
    for name, x, y in zip(NAMES[2:], one[2:], four[2:]):
        e = err_ratio(x.float().cpu(), y.float().cpu())
        print(f"  {name}: {e:.3e}", flush=True)
        assert e < 1e-3, (name, e)
    # one head against the fp64 oracle (all batches, full T)
    h = 5
    sub = [args[0][:, h:h + 1]] + [x[:, :, h:h + 1] for x in args[1:8]] + [args[8][:, h:h + 1]]
    ref = O.backward_hand(*sub)
    emu = O.emulate_bf16(*sub)
    got = [one[0][:, :, h:h + 1], one[1][:, h:h + 1], one[2][:, h:h + 1]] + [x[:, :, h:h + 1] for x in one[3:]]
    for name, a, e, g in zip(NAMES, ref, emu, got):
        assert_no_worse(f"rwkv7 full size head {h} " + name, a, e, g)


@pytest.mark.parametrize("B,T,H", [(2, 32, 2), (1, 48, 1)])
def test_rwkv7_state_only_and_stateless_ops(lib, B, T, H):
    """The siblings of the state-passing op (rwkv7_state_clampw: s0 and ds0, no final state; rwkv7_clampw: no state
    at all) are the state-passing formula with dsT = 0, respectively s0 = 0 and dsT = 0."""
    print(f"\nrwkv7 siblings B={B} T={T} H={H}", flush=True)
    s0, r, w, k, v, a, b, dy, dsT = synth.rwkv7_inputs(B, T, H, 64, seed=33)
    N = 64
    flat = lambda x: x.contiguous().view(B, T, H * N)

    # initial state only
    args = (s0, r, w, k, v, a, b, dy, torch.zeros_like(dsT))
    ref, emu = O.grads(*args), O.emulate_bf16(*args)
    t = [x.to(DEV).requires_grad_(True) for x in (s0, r, w, k, v, a, b)]
    y = R.RWKV7_STATE_CLAMPW_CUDA(t[0], *(flat(x) for x in t[1:]))
    y.backward(flat(dy.to(DEV)))
    torch.cuda.synchronize()
    got = [y.detach().view(B, T, H, N), None] + [x.grad for x in t]
    for name, a_, e, g in zip(NAMES, ref, emu, got):
        if g is not None:
            assert_no_worse("state op " + name, a_, e, g)

    # no state
    args = (torch.zeros_like(s0), r, w, k, v, a, b, dy, torch.zeros_like(dsT))
    ref, emu = O.grads(*args), O.emulate_bf16(*args)
    t = [x.to(DEV).requires_grad_(True) for x in (r, w, k, v, a, b)]
    y = R.RWKV7_CLAMPW_CUDA(*(flat(x) for x in t))
    y.backward(flat(dy.to(DEV)))
    torch.cuda.synchronize()
    got = [y.detach().view(B, T, H, N), None, None] + [x.grad for x in t]
    for name, a_, e, g in zip(NAMES, ref, emu, got):
        if g is not None:
            assert_no_worse("stateless op " + name, a_, e, g)


def test_rwkv7_long_sequence_is_no_worse_than_the_reference_kernel(lib):
    """T = 4096 on one head (the length of one call at the benchmark shape): the in-chunk inversion of the backward and the
    fp32 state must not lose accuracy with length."""
    B, T, H = 1, 4096, 1
    args = synth.rwkv7_inputs(B, T, H, 64, seed=34)
    ref = O.grads(*args)
    emu = O.emulate_bf16(*args)
    got = _run(args)
    for name, a, e, g in zip(NAMES, ref, emu, got):
        assert_no_worse("rwkv7 T4096 " + name, a, e, g)


def _fp32_inputs(B, T, H, seed):
    """The bf16 test inputs plus an fp32 perturbation below bf16 resolution, so that the fp32 mode is
    seen to read all 32 bits of every element."""
    g = torch.Generator().manual_seed(seed + 1000)
    args = synth.rwkv7_inputs(B, T, H, 64, seed=seed)
    jig = lambda x: x.float() * (1 + 1e-3 * torch.rand(x.shape, generator=g))
    s0, r, w, k, v, a, b, dy, dsT = args
    return (s0, jig(r), jig(w), jig(k), jig(v), jig(a), jig(b), jig(dy), dsT)


def assert_fp32_mode(name, ref64, emu, got):
    """fp32 mode: the error against fp64 may not exceed twice that of the reference kernel's arithmetic
    (fp32, in-chunk inversion, checkpoints every 16 steps) emulated on the CPU.  The two differ only
    in summation order, so their errors are independent samples of the same size; 2x covers that."""
    e_hip = err_ratio(ref64, got.detach().double().cpu())
    e_emu = err_ratio(ref64, emu.double())
    print(f"  {name}: hip {e_hip:.3e}  reference-kernel arithmetic {e_emu:.3e}", flush=True)
    assert e_hip <= 2.0 * e_emu + 1e-6, f"{name}: {e_hip:.3e} vs {e_emu:.3e}"
    assert e_hip < 1e-3, name                       # and far below what a bf16 rounding anywhere would leave


@pytest.mark.parametrize("B,T,H", [(2, 32, 2), (1, 256, 1)])
def test_rwkv7_fp32_mode(lib, B, T, H):
    """The reference's -D_FP32_ build (rwkv7_cuda_benchmark_state_passing.py:105-131): every tensor fp32."""
    print(f"\nrwkv7 fp32 mode B={B} T={T} H={H}", flush=True)
    args = _fp32_inputs(B, T, H, seed=35)
    ref = O.grads(*args)
    emu = O.backward_hand(*args, dtype=torch.float32, invert=True)
    got = _run(args)
    assert got[0].dtype == torch.float32 and got[3].dtype == torch.float32
    for name, a, e, g in zip(NAMES, ref, emu, got):
        assert_fp32_mode(name, a, e, g)


def test_rwkv7_fp32_mode_siblings(lib):
    B, T, H, N = 2, 32, 2, 64
    s0, r, w, k, v, a, b, dy, dsT = _fp32_inputs(B, T, H, seed=36)
    flat = lambda x: x.contiguous().view(B, T, H * N)
    args = (s0, r, w, k, v, a, b, dy, torch.zeros_like(dsT))
    ref, emu = O.grads(*args), O.backward_hand(*args, dtype=torch.float32, invert=True)
    t = [x.to(DEV).requires_grad_(True) for x in (s0, r, w, k, v, a, b)]
    y = R.RWKV7_STATE_CLAMPW_CUDA(t[0], *(flat(x) for x in t[1:]))
    y.backward(flat(dy.to(DEV)))
    torch.cuda.synchronize()
    got = [y.detach().view(B, T, H, N), None] + [x.grad for x in t]
    for name, a_, e, g in zip(NAMES, ref, emu, got):
        if g is not None:
            assert_fp32_mode("fp32 state op " + name, a_, e, g)
    args = (torch.zeros_like(s0), r, w, k, v, a, b, dy, torch.zeros_like(dsT))
    ref, emu = O.grads(*args), O.backward_hand(*args, dtype=torch.float32, invert=True)
    t = [x.to(DEV).requires_grad_(True) for x in (r, w, k, v, a, b)]
    y = R.RWKV7_CLAMPW_CUDA(*(flat(x) for x in t))
    y.backward(flat(dy.to(DEV)))
    torch.cuda.synchronize()
    got = [y.detach().view(B, T, H, N), None, None] + [x.grad for x in t]
    for name, a_, e, g in zip(NAMES, ref, emu, got):
        if g is not None:
            assert_fp32_mode("fp32 stateless op " + name, a_, e, g)


def test_rwkv7_backward_uses_the_kernel_family_of_its_forward(lib):
    """The two kernel families lay the checkpoint tensor `s` out differently and nothing in it says which one wrote it: a
    backward must run with the flags of its forward.  The wrapper keeps them on the autograd context, so a forward issued
    inside `algorithm("sweeps")` gets the step kernels' backward even when autograd runs it after the block has ended."""
    B, T, H = 2, 48, 2
    args = synth.rwkv7_inputs(B, T, H, 64, seed=35)
    ref, emu = O.grads(*args), O.emulate_bf16(*args)
    s0, r, w, k, v, a, b, dy, dsT = args
    t = [x.to(DEV).requires_grad_(True) for x in (s0, r, w, k, v, a, b)]
    with options.algorithm("sweeps"):
        y, S = R.RWKV7_STATE_PASSING_CLAMPW_CUDA(t[0], *(x.contiguous().view(B, T, H * 64) for x in t[1:]))
    assert options.current_flags() == 0                            # the block has ended: the default family is current again
    torch.autograd.backward([y, S], [dy.to(DEV).view(B, T, H * 64), dsT.to(DEV)])
    torch.cuda.synchronize()
    got = [y.detach().view(B, T, H, 64), S.detach()] + [x.grad for x in t]
    for name, a_, e, g in zip(NAMES, ref, emu, got):
        assert_no_worse("sweeps forward, backward after the block: " + name, a_, e, g)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,H", [(1, 16, 1), (2, 48, 3), (3, 160, 2)])
def test_rwkv7_forward_without_gradients_is_bit_identical(lib, B, T, H, dtype):
    """Where no backward can follow the kernels keep no states: the same outputs, bit for bit, for all three siblings, at one,
    an odd and an even number of chunks."""
    print(f"\nrwkv7 forward only B={B} T={T} H={H} {dtype}", flush=True)
    s0, r, w, k, v, a, b, _, _ = synth.rwkv7_inputs(B, T, H, 64, seed=37)
    s0 = s0.to(DEV)
    x = [t.to(DEV, dtype).view(B, T, H * 64) for t in (r, w, k, v, a, b)]
    xg = [t.clone().requires_grad_(True) for t in x]
    y, sT = R.RWKV7_STATE_PASSING_CLAMPW_CUDA(s0, *xg)
    assert y.requires_grad and sT.requires_grad
    want = [y, sT, R.RWKV7_STATE_CLAMPW_CUDA(s0, *xg), R.RWKV7_CLAMPW_CUDA(*xg)]
    for args in (x, xg):                                  # nothing asks for a gradient; gradients are off
        with torch.set_grad_enabled(args is x):
            got = [*R.RWKV7_STATE_PASSING_CLAMPW_CUDA(s0, *args), R.RWKV7_STATE_CLAMPW_CUDA(s0, *args), R.RWKV7_CLAMPW_CUDA(*args)]
        for g, e in zip(got, want):
            assert not g.requires_grad and torch.equal(g, e.detach())
    torch.cuda.synchronize()


@pytest.mark.parametrize("B,T,H", [(1, 16, 1), (2, 80, 3)])
def test_fp32_sweeps_option_runs_the_step_kernels(lib, B, T, H):
    """The option chooses the kernels in the fp32 mode too, for the backward that follows as well, and without gradients."""
    N = 64
    args = _fp32_inputs(B, T, H, 91)
    s0, r, w, k, v, a, b, dy, dsT = args
    ref = O.grads(*args)
    emu = O.backward_hand(*args, dtype=torch.float32, invert=True)
    out = {}
    for algo in ("chunked", "sweeps"):
        t = [x.to(DEV).requires_grad_(True) for x in (s0, *(x.reshape(B, T, H * N) for x in (r, w, k, v, a, b)))]
        with options.algorithm(algo):
            y, sT = R.RWKV7_STATE_PASSING_CLAMPW_CUDA(*t)
            with torch.no_grad():
                y1, sT1 = R.RWKV7_STATE_PASSING_CLAMPW_CUDA(*t)
        assert torch.equal(y, y1) and torch.equal(sT, sT1)
        g = torch.autograd.grad([y, sT], t, [dy.to(DEV).view(B, T, H * N), dsT.to(DEV)])
        out[algo] = [x.detach().double().cpu() for x in (y, sT, *g)]
        for name, want, e, got in zip(NAMES, ref, emu, out[algo]):
            assert_fp32_mode(f"{algo} {name}", want.reshape(got.shape), e.reshape(got.shape), got)
    assert not torch.equal(out["chunked"][0], out["sweeps"][0])


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("T", [16, 32, 48, 112])
@pytest.mark.parametrize("shift", [-6.0, 0.5, 6.0])
@pytest.mark.parametrize("end", [False, True])
def test_fp32_results_keep_24_bits(lib, T, f32, shift, end):
    """One, two, three and seven chunks, slow to strong decays, with and without a gradient of the final state: every fp32 result (y and
    the gradients are fp32 in the fp32 mode alone) against the step form in 64 bits.  Bound: each factor, sum and product of a chunk
    leaves about half a unit in the last place, 2^-24, four to eight of them in a result: 4e-7.  (Products without their second-order
    terms, m m', h l', l h', would leave 4.5e-6.)  dw = G sig (1 - sig): G is a difference that is carried through the call, 3e-7 a
    chunk at most, adding up as a random walk; 1 - sig is rounded at 2^-25 and about e^-w."""
    B, H, N = 2, 3, 64
    g = torch.Generator().manual_seed(T)
    n = lambda *s: torch.randn(*s, generator=g)
    kk = torch.nn.functional.normalize(n(B, T, H, N), dim=-1)
    s0, dsT = n(B, H, N, N) * 0.1, n(B, H, N, N) * 0.1
    x = [n(B, T, H, N) * 0.5, n(B, T, H, N) + shift, n(B, T, H, N) * 0.5, n(B, T, H, N) * 0.5, -kk, kk * torch.sigmoid(n(B, T, H, N)), n(B, T, H, N)]
    x = [t.to(torch.float32 if f32 else torch.bfloat16) for t in x]
    S, r, w, k, v, a, b = p = [t.double().requires_grad_(True) for t in (s0, *x[:6])]
    d = torch.exp(-math.exp(-0.5) * torch.sigmoid(w))
    ys, sas = [], []
    for t in range(T):
        sas.append((S * a[:, t, :, None, :]).sum(-1))
        S = S * d[:, t, :, None, :] + sas[-1][..., None] * b[:, t, :, None, :] + v[:, t, :, :, None] * k[:, t, :, None, :]
        ys.append((S * r[:, t, :, None, :]).sum(-1))
    y = torch.stack(ys, 1)
    grads = torch.autograd.grad([y, S] if end else [y], p, [x[6].double(), dsT.double()] if end else [x[6].double()])
    want = dict(zip(("y", "sT", "sa", "ds0", "dr", "dw", "dk", "dv", "da", "db"), (y.detach(), S.detach(), torch.stack(sas, 1).detach(), *grads)))
    dev = [t.to(DEV) for t in (s0, *x)]
    new = lambda *s: torch.full(s, math.nan, device=DEV)
    like = lambda: torch.full_like(dev[1], math.nan)
    got = dict(y=like(), sT=new(B, H, N, N), s=new(B, H, T // 16, N, N), sa=new(B, T, H, N), ds0=new(B, H, N, N), **{z: like() for z in ("dr", "dw", "dk", "dv", "da", "db")})
    sfx = "_f32" if f32 else ""
    call(f"rwkv7_statepassing_forward{sfx}_ex", DEV, B, T, H, *dev[:7], got["y"], got["sT"], got["s"], got["sa"], 0)
    call(f"rwkv7_statepassing_backward{sfx}_ex", DEV, B, T, H, *dev[1:], dsT.to(DEV) if end else None, got["s"], got["sa"],
         *(got[z] for z in ("ds0", "dr", "dw", "dk", "dv", "da", "db")), 0)
    with torch.no_grad():                                   # the forward that keeps nothing: the same bits
        y1, sT1 = R.RWKV7_STATE_PASSING_CLAMPW_CUDA(dev[0], *(t.view(B, T, H * N) for t in dev[1:7]))
    assert torch.equal(y1.view_as(got["y"]), got["y"]) and torch.equal(sT1, got["sT"])
    for z, q in want.items():
        e = ((got[z].double().cpu() - q).norm() / q.norm()).item()
        print(f"  {z}: {e:.2e}", flush=True)
        dw = 3e-7 * max(1.0, T / 16) ** 0.5 * 2 + 2.0 ** -25 * math.exp(shift + 1)
        assert e <= (2.0 ** -8 if got[z].dtype == torch.bfloat16 else dw if z == "dw" else 4e-7), (z, e)


FLT_MAX = torch.finfo(torch.float32).max


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("f32,name,t", [(False, "s0", 3), (False, "dsT", 3), (True, "s0", 3), (True, "dsT", 3), (True, "r", 23), (True, "k", 23), (True, "v", 16),
                                        (True, "v", 31), (True, "b", 23), (True, "dy", 16), (True, "dy", 31)])
def test_finite_values_beyond_the_largest_bf16(f32, name, t, sign):
    """The largest fp32 value as one element of an input (s0 and dsT are fp32 in either mode): results are finite where the step form's
    are in fp32, and as accurate as without it.  Bound of an fp32 result: one element carries the norm, so its roundings do not average out;
    32 of them at 2^-24 (decays over 48 steps, sums and splits).  A bf16 result: its own rounding."""
    B, T, H, N = 1, 48, 1, 64
    s0, r, w, k, v, a, b, dy, dsT = synth.rwkv7_inputs(B, T, H, N, seed=7)
    x = dict(s0=s0, r=r, w=w, k=k, v=v, a=a, b=b, dy=dy, dsT=dsT)
    dt = torch.float32 if f32 else torch.bfloat16
    x = {n: (z if n == "w" else z * 2.0 ** -9).to(z.dtype if n in ("s0", "dsT") else dt) for n, z in x.items()}          # no product overflows
    if name in ("s0", "dsT"):
        x[name][0, 0, t, 5] = sign * FLT_MAX
    else:
        x[name][0, t, 0, 5] = sign * FLT_MAX
    args = [x[n] for n in ("s0", "r", "w", "k", "v", "a", "b", "dy", "dsT")]
    ref = O.grads(*args)
    assert all(float(z.abs().max()) < FLT_MAX * 1.0001 for z in ref)
    got = _run(args)
    for n, want, g in zip(NAMES, ref, got):
        assert bool(g.isfinite().all()), n
        e = ((g.double().cpu() - want).norm() / want.norm()).item()
        print(f"  {n}: {e:.2e}", flush=True)
        assert e <= (2.0 ** -19 if g.dtype == torch.float32 else 2.0 ** -8), (n, e)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_no_decay_has_no_decay_gradient(lib, dtype):
    """w = -inf, or so low that e^-w overflows: sigmoid(w) is zero, the step keeps the state, and dw is zero and not merely small; where
    sigmoid(w) is subnormal (spacing 2^-149, so 2^-22 of 4e-39) dw is still right."""
    B, T, H, N = 1, 32, 2, 64
    s0, r, w, k, v, a, b, dy, dsT = synth.rwkv7_inputs(B, T, H, N, seed=8)
    w[:, 3, :, 7], w[:, 16, :, 8], w[:, 31, :, 9] = -math.inf, -120.0, -3e38
    w[:, 7], w[:, 20] = -88.5, -87.5          # (bf16 holds both)
    off = w < -100
    args = [s0, *(x.to(dtype) for x in (r, w, k, v, a, b, dy)), dsT]
    got = _run(args)
    assert float(got[NAMES.index("dw")].cpu()[off].abs().max()) == 0.0
    ref = O.grads(*args)
    dw, want = got[NAMES.index("dw")].double().cpu(), ref[NAMES.index("dw")]
    rel, spacing = (2e-5, 2.0 ** -149) if dtype == torch.float32 else (2.0 ** -8, 2.0 ** -133)        # (of subnormal results)
    for t in (7, 20):
        assert float((dw[:, t] - want[:, t]).norm()) <= rel * float(want[:, t].norm()) + spacing * math.sqrt(want[:, t].numel()), t
    emu = O.emulate_bf16(*args) if dtype == torch.bfloat16 else O.backward_hand(*args, dtype=torch.float32)
    for name, x, e, g in zip(NAMES, ref, emu, got):
        if dtype == torch.bfloat16:
            assert_no_worse(name, x, e, g)
        else:
            assert_fp32_mode(name, x, e, g)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", ["r", "k", "v", "a", "b", "s0"])
@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
def test_where_an_infinity_reaches(lib, dtype, name, value):
    """One infinity or NaN among the inputs: what is not finite in the step form is not finite here (NaN where that has an infinity, as the
    header says), nothing before its chunk is touched, and neither are other heads and batch rows, gradients included."""
    B, T, H, N = 2, 48, 2, 64
    s0, r, w, k, v, a, b, dy, dsT = synth.rwkv7_inputs(B, T, H, N, seed=9)
    x = dict(s0=s0, r=r, w=w, k=k, v=v, a=a, b=b, dy=dy, dsT=dsT)
    x = {n: z.to(torch.float32 if n in ("s0", "dsT") else dtype) for n, z in x.items()}
    clean = _run(list(x.values()))
    x[name] = x[name].clone()
    if name == "s0":
        x[name][0, 0, 3, 5] = value
    else:
        x[name][0, 23, 0, 5] = value
    got = _run(list(x.values()))
    step = O.recurrent(*(x[n].double() for n in ("s0", "r", "w", "k", "v", "a", "b")))
    for want, g in zip(step, got):
        assert not bool((~want.isfinite() & g.cpu().isfinite()).any())
    assert not bool(got[0][0, 23, 0].isfinite().all())
    if name != "s0":
        assert torch.equal(got[0][:, :16], clean[0][:, :16])
    for n, c, g in zip(NAMES, clean, got):
        per_head = (lambda z: z) if n in ("sT", "ds0") else (lambda z: z.transpose(1, 2))         # [B, H, ...]
        c, g = per_head(c), per_head(g)
        assert torch.equal(c[1], g[1]) and torch.equal(c[0, 1], g[0, 1]), n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("c", [-8.0, -5.0, -2.0, 2.0])
def test_rwkv7_the_decay_of_a_chunk_is_within_half_a_place(lib, c, dtype):
    """One chunk, all other inputs zero, states of ones: sT and ds0 are the chunk's decay as the kernels multiply states by it.  Where it is
    slow its rounding is what adds up over a sequence.  Bound: half a place of the result, and of the exponent 2^-20 for the steps' sigmoids
    (argument of up to 14 rounded 3.3e-7, its constant 1.4e-7, exponential, sum, reciprocal and product 4e-7) and for the series."""
    B, T, H, N = 1, 16, 64, 64
    g = torch.Generator().manual_seed(int(10 - 10 * c))
    w = (c + 0.5 * torch.randn(B, T, H, N, generator=g)).to(dtype).to(DEV)
    zero, one, f32 = torch.zeros_like(w), torch.ones(B, H, N, N, device=DEV), int(dtype == torch.float32)
    y, sT, s, sa = torch.empty_like(w), torch.empty_like(one), torch.empty_like(one), torch.empty(B, T, H, N, device=DEV)
    call("rwkv7_forward_ws", y.device, B, T, H, f32, one, zero, w, zero, zero, zero, zero, y, sT, s, sa, None, 0)
    ds0, d = torch.empty_like(one), [torch.empty_like(w) for _ in range(6)]
    call("rwkv7_backward_ws", y.device, B, T, H, f32, zero, w, zero, zero, zero, zero, zero, one, s, sa, ds0, *d, None, 0)
    e = -0.6065306597 * torch.sigmoid(w.double()).sum(1)[:, :, None, :]
    place = torch.exp2(torch.floor(e / math.log(2)) - 23)
    for name, x in (("sT", sT), ("ds0", ds0)):
        off = (x.double() - e.exp()).abs()
        print(f"  {name}: {float((off / place).max()):.3f} places", flush=True)
        assert bool((off <= 0.5 * place - e * e.exp() * 2.0 ** -20).all()), name


def test_rwkv7_more_heads_than_one_launch_takes(lib):
    """8.4 million heads of 16 tokens: 512 work items each are more than the 2^32 that a launch may have along x (beyond, it runs the remainder
    of 2^32 and reports nothing).  One tensor (17 GB) is all six inputs; the rows at
    either end and at the border of the launches have the bits of a call of their own."""
    B, T, H, N = 32768, 16, 257, 64
    g = torch.Generator().manual_seed(3)
    x = (torch.randn(1, T, H * N, generator=g) * 0.1).to(torch.bfloat16).to(DEV).repeat(B, 1, 1)
    rows = [0, 16319, 16320, 16321, 32640, 32641, 32767]      # (2^22 heads: within row 16320)
    for i in rows:
        x[i] = (torch.randn(T, H * N, generator=g) * 0.1).to(torch.bfloat16).to(DEV)
    y = torch.empty_like(x)
    call("rwkv7_forward_ws", y.device, B, T, H, 0, None, x, x, x, x, x, x, y, None, None, None, None, 0)
    few, want = x[rows].contiguous(), torch.empty(len(rows), T, H * N, dtype=torch.bfloat16, device=DEV)
    call("rwkv7_forward_ws", y.device, len(rows), T, H, 0, None, few, few, few, few, few, few, want, None, None, None, None, 0)
    same = [torch.equal(y[i], z) for i, z in zip(rows, want)] + [torch.equal(y[1], y[-3])]
    assert all(same), same
