"""What the speed of this framework is measured on: its operators as a training or serving program calls them.

A case is a dict of plain values.  `op` names the operator (a module of rwkv_cuda_amd, rwkv7 in its three variants),
`train` says whether a pass is forward + backward or forward alone, the rest are sizes.  All inputs live in GPU memory and
are drawn there from the seed, with the distributions of the operators' own checks and benchmarks.
"""
import math

import torch

from rwkv_cuda_amd import depthwise_conv1d, rwkv7_fast_fused, wkv, wkv5, wkv5_bf16, wkv5a, wkv6, wkv6_state

DEV = "cuda"
BF16_OPS = ("wkv5_bf16", "wkv6", "wkv6_state")
FP32_OPS = ("wkv5", "wkv5a")


def listed():
    return [
        # RWKV-4, one GPU's micro-batch of a small model: two short launches, so the calls themselves count
        dict(name="wkv4_small", op="wkv", B=4, T=512, C=768, train=True),
        # RWKV-4 at the batch and length of the operator's own check
        dict(name="wkv4_batch", op="wkv", B=32, T=768, C=768, train=True),
        # depthwise_conv1d at the shape its published timings are quoted on
        dict(name="conv", op="depthwise_conv1d", B=32, C=768, T=768, train=True),
        # the same operator at a batch and a length that are no multiples of anything but the required 4
        dict(name="conv_ragged", op="depthwise_conv1d", B=13, C=384, T=1500, train=True),
        # RWKV-5 layer, head size 64
        dict(name="wkv5", op="wkv5_bf16", B=8, T=4096, H=32, N=64, train=True),
        # RWKV-5 layer with the heads of 128 channels that its driver ships with
        dict(name="wkv5_n128", op="wkv5_bf16", B=8, T=4096, H=32, N=128, train=True),
        # RWKV-5 in fp32, the precision of its first driver, at that driver's benchmark shape
        dict(name="wkv5_fp32", op="wkv5", B=8, T=4096, H=64, N=64, train=True),
        # RWKV-6 layer: the headline shape
        dict(name="wkv6", op="wkv6", B=8, T=4096, H=32, N=64, train=True),
        # RWKV-6 fine-tuning on one document: a single sequence of no round length, with its initial state
        dict(name="wkv6_state_one", op="wkv6_state", B=1, T=3001, H=32, N=64, train=True),
        # RWKV-7 layer, a long sequence as four calls that pass the state on
        dict(name="rwkv7", op="rwkv7", variant="passing", dtype="bf16", B=8, T=1024, calls=4, H=64, N=64, train=True),
        # RWKV-7 in fp32, one call
        dict(name="rwkv7_fp32", op="rwkv7", variant="passing", dtype="fp32", B=8, T=1024, calls=1, H=64, N=64, train=True),
        # RWKV-7 serving: the next 16 tokens of one conversation
        dict(name="rwkv7_next16", op="rwkv7", variant="passing", dtype="bf16", B=1, T=16, calls=1, H=32, N=64, train=False),
    ]


# a drawn case has no more tokens x channels, and no more multiply-adds of a convolution, than these
MAX_ELEMS = 8 * 4096 * 4096
MAX_CONV_MACS = 13 * 384 * 1500 * 1500


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["wkv", "depthwise_conv1d", "wkv5_bf16", "wkv5_bf16", "wkv5", "wkv5a", "wkv6", "wkv6", "wkv6_state", "rwkv7", "rwkv7"])
    train = rng.random() < 0.75
    while True:
        B = _log_int(rng, 1, 32)
        if op == "wkv":
            case = dict(op=op, B=B, T=_log_int(rng, 16, 4096), C=_log_int(rng, 64, 2560))
        elif op == "depthwise_conv1d":
            case = dict(op=op, B=B, C=_log_int(rng, 64, 1024), T=4 * _log_int(rng, 8, 1024))
            if B * case["C"] * case["T"] ** 2 > MAX_CONV_MACS:
                continue
        elif op == "rwkv7":
            T = 16 * _log_int(rng, 1, 256)
            calls = rng.choice([1, 2, 4]) if T <= 1024 else 1
            variant = rng.choice(["passing", "state", "none"])
            case = dict(op=op, variant=variant, dtype=rng.choice(["bf16", "bf16", "fp32"]), B=B, T=T,
                        calls=calls if variant == "passing" else 1, H=_log_int(rng, 8, 64), N=64)
        else:
            N = 128 if op == "wkv5_bf16" and rng.random() < 0.4 else 64
            case = dict(op=op, B=B, T=_log_int(rng, 16, 8192), H=_log_int(rng, 8, 64), N=N)
        # fp32 elements are twice the bytes; one of rwkv7 takes about as much arithmetic as two of the others
        weight = (2 if op in FP32_OPS or op == "rwkv7" else 1) * (2 if case.get("dtype") == "fp32" else 1)
        if _elems(case) * weight <= MAX_ELEMS:
            case["train"] = train
            return case


def _elems(case):
    C = case["C"] if "C" in case else case["H"] * case["N"]
    return case["B"] * case["T"] * case.get("calls", 1) * C


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    normal = lambda *s: torch.randn(*s, generator=g, device=DEV)
    uniform = lambda lo, hi, *s: torch.rand(*s, generator=g, device=DEV) * (hi - lo) + lo
    op, B, T = case["op"], case["B"], case["T"]
    C = case["C"] if "C" in case else case["H"] * case["N"]
    H, N = case.get("H"), case.get("N")
    bf = torch.bfloat16
    if op == "wkv":
        args = [normal(C) * 0.5, normal(C) * 0.5, normal(B, T, C).clamp_(-8, 8), normal(B, T, C)]
        up = [normal(B, T, C)]
    elif op == "depthwise_conv1d":
        args = [normal(C, T) / math.sqrt(T), normal(B, C, T)]
        up = [normal(B, C, T)]
    elif op in BF16_OPS:
        args = [(normal(B, T, C) * 0.5).to(bf) for _ in range(3)]
        args.append((normal(H, N) * 0.5 - 0.5).to(bf) if op == "wkv5_bf16" else (normal(B, T, C) * 0.7 - 0.6).to(bf))
        args.append((normal(H, N) * 0.3).to(bf))
        if op == "wkv6_state":
            args.append((normal(B, H, N, N) * 0.1).to(bf))
        up = [normal(B, T, C).to(bf)]
    elif op == "wkv5":
        args = [uniform(-1, 1, B, T, C) for _ in range(3)] + [uniform(-1, 1, C) for _ in range(2)]
        up = [uniform(-1, 1, B, T, C)]
    elif op == "wkv5a":
        args = [uniform(-1, 1, B, T, C) for _ in range(3)]
        args += [uniform(lo, 1, H, N) for lo in (-8, -1, -8, -1)]        # w1, u1, w2, u2
        up = [uniform(-1, 1, B, T, C)]
    else:
        dt = torch.float32 if case["dtype"] == "fp32" else bf
        args, up = [], []
        if case["variant"] != "none":
            args.append(normal(B, H, N, N) * 0.1)
        for _ in range(case["calls"]):
            r, k, v = (normal(B, T, C) * 0.5 for _ in range(3))
            w = normal(B, T, C) + 0.5
            kk = torch.nn.functional.normalize(normal(B, T, H, N), dim=-1)
            a, b = -kk, kk * torch.sigmoid(normal(B, T, H, N))
            args += [x.to(dt).view(B, T, C) for x in (r, w, k, v, a, b)]
            up.append(normal(B, T, C).to(dt))
        if case["variant"] == "passing":
            up.append(normal(B, H, N, N) * 0.1)                          # the gradient that comes back for the final state
    if case["train"]:
        for x in args:
            x.requires_grad_(True)
    return dict(case=case, args=args, up=up)


def _forward(case, args):
    """The operator's outputs, in the order of the upstream gradients."""
    op, B, T = case["op"], case["B"], case["T"]
    C = case["C"] if "C" in case else case["H"] * case["N"]
    if op == "wkv":
        return [wkv.RUN_CUDA(B, T, C, *args)]
    if op == "depthwise_conv1d":
        return [depthwise_conv1d.RUN_CUDA(*args, B, C, T, 0.0)]
    if op == "wkv5a":
        return [wkv5a.CUDA_1(*args)]
    if op in ("wkv5_bf16", "wkv5", "wkv6", "wkv6_state"):
        module = {"wkv5_bf16": wkv5_bf16, "wkv5": wkv5, "wkv6": wkv6, "wkv6_state": wkv6_state}[op]
        return [module.RUN_CUDA(B, T, C, case["H"], *args)]
    if case["variant"] == "none":
        return [rwkv7_fast_fused.RWKV7_CLAMPW_CUDA(*args)]
    if case["variant"] == "state":
        return [rwkv7_fast_fused.RWKV7_STATE_CLAMPW_CUDA(*args)]
    state, out = args[0], []
    for i in range(case["calls"]):
        y, state = rwkv7_fast_fused.RWKV7_STATE_PASSING_CLAMPW_CUDA(state, *args[1 + 6 * i:7 + 6 * i])
        out.append(y)
    return out + [state]


def run(state):
    case, args = state["case"], state["args"]
    if not case["train"]:
        with torch.no_grad():
            return _forward(case, args)
    out = _forward(case, args)
    grads = torch.autograd.grad(out, args, state["up"])
    return [x.detach() for x in out] + list(grads)


def work(case):
    """Inputs and outputs of each direction moved once; the multiply-adds of the operator's defining recurrence."""
    op, train, n = case["op"], case["train"], _elems(case)
    if op == "wkv":
        # a step has two exponentials, four products and a division; backward about twice that
        return {"bytes": 4 * n * (3 + (5 if train else 0)), "flops": n * (20 + (50 if train else 0))}
    if op == "depthwise_conv1d":
        macs = case["B"] * case["C"] * case["T"] * (case["T"] + 1) // 2
        weights = 4 * case["C"] * case["T"]
        return {"bytes": 4 * n * (2 + (3 if train else 0)) + weights * (1 + (2 if train else 0)), "flops": 2 * macs * (3 if train else 1)}
    states = case["B"] * case["H"] * case["N"] ** 2
    if op == "rwkv7":
        eb = 4 if case["dtype"] == "fp32" else 2
        state_tensors = {"none": 0, "state": 1, "passing": 2}[case["variant"]] * (2 if train else 1)
        # per state element and token: two products with vectors, the decay and two outer products; backward about twice that
        return {"bytes": eb * n * (7 + (13 if train else 0)) + 4 * states * state_tensors, "flops": n * case["N"] * (9 + (20 if train else 0))}
    eb = 4 if op in FP32_OPS else 2
    per_token = (1 if op in ("wkv6", "wkv6_state") else 0)               # the decay is a tensor with a gradient
    tensors = 4 + per_token + (7 + 2 * per_token if train else 0)
    state_bytes = 2 * states * (3 if train else 1) if op == "wkv6_state" else 0
    # per state element and token: the outer product, the decay, the product with r; backward four products and two updates
    return {"bytes": eb * n * tensors + state_bytes, "flops": n * case["N"] * (5 + (14 if train else 0))}


# About four times the largest relative error seen in any output and gradient.  fp32 operators: against the same path in 64
# bits (wkv 2e-7, depthwise_conv1d 6e-7, wkv5 6e-7; wkv5a 1e-5, since its slow decays are rounded to fp32 before they act
# thousands of times; rwkv7 1e-5, since a backward may rebuild states by division).  bf16 operators: two algorithms of the
# framework against each other, i.e. values that fall on the other side of a rounding (wkv6 4e-4, rwkv7 1.6e-4; wkv5 2e-3,
# its decay gradient being a sum over the batch of rounded rows).
TOLERANCE = {"wkv": 1e-6, "depthwise_conv1d": 3e-6, "wkv5": 3e-6, "wkv5a": 5e-5, "rwkv7 fp32": 5e-5,
             "wkv6": 2e-3, "wkv6_state": 2e-3, "wkv5_bf16": 8e-3, "rwkv7 bf16": 1e-3}


def tolerance(case):
    return {"rel": TOLERANCE[case["op"] + (" " + case["dtype"] if "dtype" in case else "")]}
