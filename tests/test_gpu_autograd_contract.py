"""GPU: what a program around the operators relies on, beside the numbers: checkpoints and saved-tensor hooks, shapes of gradients,
what is refused and with which error."""
import pytest
import torch
from torch.utils.checkpoint import checkpoint

from rwkv_cuda_amd import depthwise_conv1d, rwkv7_fast_fused as R, synth, wkv, wkv5, wkv5_bf16, wkv5a, wkv6, wkv6_state
from rwkv_cuda_amd._lib import RwkvHipError
from _gpu_util import DEV

pytestmark = pytest.mark.gpu
B, T, H = 2, 48, 2
C = H * 64


def _f32(*shape, seed=0):
    return torch.rand(*shape, generator=torch.Generator().manual_seed(seed)) * 2 - 1


def _case(op):
    """(function of the tensors, tensors)"""
    if op == "wkv":
        w, u, k, v, _ = synth.wkv4_inputs(B, T, C, seed=1)
        return lambda *x: wkv.RUN_CUDA(B, T, C, *x), [w, u, k, v]
    if op == "depthwise_conv1d":
        w, k, _ = synth.timex_inputs(B, C, T, seed=2)
        return lambda *x: depthwise_conv1d.RUN_CUDA(*x, B, C, T, 0.5), [w, k]
    if op == "wkv5":
        return lambda *x: wkv5.RUN_CUDA(B, T, C, H, *x), [_f32(B, T, C, seed=i) for i in range(3)] + [_f32(C, seed=3), _f32(C, seed=4)]
    if op == "wkv5a":
        return wkv5a.CUDA_1, [_f32(B, T, C, seed=i) for i in range(3)] + [_f32(H, 64, seed=3 + i) for i in range(4)]
    if op in ("wkv5_bf16", "wkv5_bf16_128"):
        h = H if op == "wkv5_bf16" else H // 2
        return lambda *x: wkv5_bf16.RUN_CUDA(B, T, C, h, *x), list(synth.wkv5_inputs(B, T, C, h, seed=5)[:5])
    if op == "wkv6":
        return lambda *x: wkv6.RUN_CUDA(B, T, C, H, *x), list(synth.wkv6_inputs(B, T, C, H, seed=6)[:5])
    if op == "wkv6_state":
        r, k, v, w, u, _, s0 = synth.wkv6_inputs(B, T, C, H, seed=7, state=True)
        return lambda *x: wkv6_state.RUN_CUDA(B, T, C, H, *x), [r, k, v, w, u, s0]
    s0, r, w, k, v, a, b, _, _ = synth.rwkv7_inputs(B, T, H, 64, seed=8)
    x = [t.to(torch.float32 if op.endswith("f32") else torch.bfloat16).view(B, T, C) for t in (r, w, k, v, a, b)]
    if "none" in op:
        return R.RWKV7_CLAMPW_CUDA, x
    if "passing" in op:
        return R.RWKV7_STATE_PASSING_CLAMPW_CUDA, [s0] + x
    return R.RWKV7_STATE_CLAMPW_CUDA, [s0] + x


OPS = ["wkv", "depthwise_conv1d", "wkv5", "wkv5a", "wkv5_bf16", "wkv5_bf16_128", "wkv6", "wkv6_state",
       "rwkv7_none", "rwkv7_state", "rwkv7_passing", "rwkv7_passing_f32"]


def _grads(out, t):
    out = out if isinstance(out, tuple) else (out,)
    up = [torch.ones_like(o) for o in out]
    return [o.detach() for o in out] + list(torch.autograd.grad(out, t, up))


@pytest.mark.parametrize("op", OPS)
def test_checkpoint_and_saved_tensor_hooks(lib, op):
    """The gradients under a checkpoint without re-entry are those without, and every saved tensor is unpacked once."""
    f, x = _case(op)
    t = [z.to(DEV).requires_grad_(True) for z in x]
    want = _grads(f(*t), t)
    got = _grads(checkpoint(f, *t, use_reentrant=False), t)
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    count = {}

    def pack(z):
        count[len(count)] = 0
        return len(count) - 1, z

    def unpack(p):
        count[p[0]] += 1
        return p[1]

    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        out = f(*t)
    got = _grads(out, t)
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    assert count and all(n == 1 for n in count.values()), count


@pytest.mark.parametrize("op", ["rwkv7_none", "rwkv7_state", "rwkv7_passing", "rwkv7_passing_f32"])
def test_rwkv7_gradients_have_the_shapes_of_their_inputs(lib, op):
    """The functions take r as [B,T,C]; the others may be [B,T,H,64] as well, the same memory."""
    f, x = _case(op)
    want = _grads(f(*(t := [z.to(DEV).requires_grad_(True) for z in x])), t)
    first = len(x) - 6
    y = [z.view(B, T, H, 64) if i in (first + 1, first + 4) else z for i, z in enumerate(x)]
    got = _grads(f(*(t := [z.to(DEV).requires_grad_(True) for z in y])), t)
    n = len(want) - len(x)
    for a, b, z in zip(want[n:], got[n:], y):
        assert b.shape == z.shape and torch.equal(a.reshape(z.shape), b)


def test_rwkv7_functions_and_classes_take_r_in_their_own_shape(lib):
    for op, cls in (("rwkv7_none", R.RWKV7_CLAMPW_CUDA_OP), ("rwkv7_state", R.RWKV7_STATE_CLAMPW_CUDA_OP), ("rwkv7_passing", R.RWKV7_STATE_PASSING_CLAMPW_CUDA_OP)):
        f, x = _case(op)
        t = [z.to(DEV) for z in x]
        n = len(t) - 6
        heads = t[:n] + [z.view(B, T, H, 64) for z in t[n:]]
        y, z = f(*t), cls.apply(*heads)
        y, z = (y[0], z[0]) if op == "rwkv7_passing" else (y, z)
        assert y.shape == (B, T, C) and z.shape == ((B, T, C) if op == "rwkv7_passing" else (B, T, H, 64)) and torch.equal(y, z.view(B, T, C))
        for call, args in ((f, heads), (cls.apply, t)):
            with pytest.raises((AssertionError, ValueError)):
                call(*args)


@pytest.mark.parametrize("op", ["wkv5", "wkv5a"])
def test_fp32_decays_of_any_alignment(lib, op):
    """A decay may be a view at an odd offset of a larger parameter."""
    f, x = _case(op)
    want = _grads(f(*(t := [z.to(DEV).requires_grad_(True) for z in x])), t)
    t = []
    for i, z in enumerate(x):
        z = z.to(DEV)
        if i in (3, 5):
            z = torch.cat([z.new_zeros(1), z.reshape(-1)])[1:].view(z.shape)
            assert z.data_ptr() % 16 == 4
        t.append(z.requires_grad_(True))
    got = _grads(f(*t), t)
    assert all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.parametrize("op", OPS)
def test_errors_of_either_direction_are_the_packages_own(lib, op):
    """No tokens, and an upstream gradient off the 16-byte grid: refused by the host code, in the backward on a thread of the engine."""
    f, x = _case(op)
    t = [z.to(DEV).requires_grad_(True) for z in x]
    out = f(*t)
    out = out if isinstance(out, tuple) else (out,)
    up = [torch.ones_like(o) for o in out]
    up[0] = torch.cat([up[0].new_zeros(1), up[0].reshape(-1)])[1:].view(up[0].shape)
    assert up[0].data_ptr() % 16 != 0
    with pytest.raises(RwkvHipError, match="align"):
        torch.autograd.grad(out, t, up)
    if op.startswith(("wkv5", "wkv6")) and op != "wkv5a":
        empty = [z.detach()[:, :0].contiguous() if z.dim() == 3 else z.detach() for z in t]
        module, h = {"wkv5": (wkv5, H), "wkv5_bf16": (wkv5_bf16, H), "wkv5_bf16_128": (wkv5_bf16, H // 2), "wkv6": (wkv6, H), "wkv6_state": (wkv6_state, H)}[op]
        with pytest.raises(RwkvHipError):
            module.RUN_CUDA(B, 0, C, h, *empty)
