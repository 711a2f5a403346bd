"""GPU: depthwise_conv1d at the lengths and batch sizes that are not whole tiles (timex_conv_any, timex_gw_any, timex_gw_short), against the fp64
oracle: one block of steps, a block and a piece, odd numbers of blocks, the longest sequence, batches of one row up to more than
one unit, batch groups that are summed by a second kernel and ones that are not.

Tolerance: the fp32 ops' bar of 1e-5, and element by element the bound of an fp32 loop: n products leave at most n 2^-24 of the
sum of their magnitudes.  An operand keeps its 24 bits, a product loses less than 2^-23, and a matrix instruction adds up to 32 products
at a time in six parts: fewer roundings than the loop has."""
import pytest
import torch

from oracle import err_ratio, max_rel_to_peak
from oracle import timex as OT
from rwkv_cuda_amd import depthwise_conv1d, synth
from rwkv_cuda_amd._call import call
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


@pytest.mark.parametrize("T", [4, 8, 28, 32, 36, 60, 100, 384, 388, 516, 1000, 1028, 1056, 1500, 2048, 2052, 4092, 4096])
@pytest.mark.parametrize("B", [1, 2, 5, 13])
def test_shapes(lib, B, T):
    print(f"\ntimex any B={B} T={T}", flush=True)
    _check(B, 3, T, *synth.timex_inputs(B, 3, T, seed=B + T))


@pytest.mark.parametrize("B,C,T", [(7, 5, 96), (16, 2, 772), (31, 2, 68), (32, 3, 100), (33, 2, 36), (64, 1, 1500), (70, 2, 4), (3, 600, 52),
                                   (13, 40, 500), (33, 40, 500), (13, 200, 100), (7, 40, 1500)])   # the last four: units of unequal numbers of rows
def test_more_batches(lib, B, C, T):
    print(f"\ntimex any B={B} C={C} T={T}", flush=True)
    _check(B, C, T, *synth.timex_inputs(B, C, T, seed=B + C + T))


def test_reference_signature_gives_per_batch_kernel_gradients(lib):
    B, C, T = 3, 4, 76
    w, k, g = synth.timex_inputs(B, C, T, seed=9)
    d = [x.to(DEV) for x in (w, k, g)]
    gw, gk = torch.empty(B, C, T, device=DEV), torch.empty(B, C, T, device=DEV)
    call("rwkv_timex_backward", d[0].device, *d, gw, gk, B, C, T)
    ref_gw, ref_gk = OT.grads_closed_form(*(x.double() for x in (w, k, g)), B, C, T)
    assert max_rel_to_peak(ref_gw, gw.double().cpu()) <= 1e-5 and max_rel_to_peak(ref_gk, gk.double().cpu()) <= 1e-5


def _some_channels(B, C, T, seed, some):
    """w, k, g on the GPU, and out, gw, gk of a few channels in 64 bits."""
    w, k, g = synth.timex_inputs(B, C, T, seed=seed)
    return [x.to(DEV) for x in (w, k, g)], OT.grads(w[some], k[:, some], g[:, some], B, len(some), T)


@pytest.mark.parametrize("B,C,T", [(32, 520, 36), (16, 520, 132), (13, 1030, 68), (9, 520, 292), (3, 768, 388), (16, 520, 500), (5, 540, 452), (24, 600, 484)])
def test_many_short_rows(lib, B, C, T):
    """More workgroups than the card takes at a time, a wave a column tile (one tile to eight; units of unequal numbers of rows)."""
    some = [0, C // 2, C - 1]
    (w, k, g), ref = _some_channels(B, C, T, B + T, some)
    w, k = w.requires_grad_(True), k.requires_grad_(True)
    x = depthwise_conv1d.RUN_CUDA(w, k, B, C, T, 0.0)
    gw, gk = torch.autograd.grad(x, (w, k), g)
    for name, a, got in zip(("x", "gw", "gk"), ref, (x[:, some], gw[some], gk[:, some])):
        assert max_rel_to_peak(a, got.detach().double().cpu()) <= 1e-5, name


@pytest.mark.parametrize("B,C,T", [(3, 700, 1500), (3, 384, 1500), (10, 330, 1300), (19, 350, 772), (13, 320, 644)])
def test_last_rounds_of_few_units(lib, B, C, T):
    """Units chosen with a last round that leaves CUs one workgroup (the second: not), of one size and of two."""
    some = [0, C // 2, C - 1]
    (w, k, g), ref = _some_channels(B, C, T, B + T, some)
    w, k = w.requires_grad_(True), k.requires_grad_(True)
    x = depthwise_conv1d.RUN_CUDA(w, k, B, C, T, 0.0)
    gw, gk = torch.autograd.grad(x, (w, k), g)
    for name, a, got in zip(("x", "gw", "gk"), ref, (x[:, some], gw[some], gk[:, some])):
        assert max_rel_to_peak(a, got.detach().double().cpu()) <= 1e-5, name


@pytest.mark.parametrize("B,C,T", [(24, 300, 508), (27, 300, 452), (12, 768, 452), (32, 64, 512 + 4), (6, 200, 644), (16, 64, 708), (16, 64, 712)])
def test_kernel_gradients_of_middle_lengths(lib, B, C, T):
    """Lag tiles of 32 or of 256, and as many parts of the batch, as take less time: either side of the lengths where the rule changes."""
    some = [0, C // 2, C - 1]
    (w, k, g), ref = _some_channels(B, C, T, B + T, some)
    n = lib.rwkv_timex_backward_ws_bytes(B, C, T)
    gw, gk = _backward_ws(w, k, g, B, C, T, torch.empty(max(n, 16), dtype=torch.uint8, device=DEV), n)
    assert max_rel_to_peak(ref[1], gw[some].double().cpu()) <= 1e-5 and max_rel_to_peak(ref[2], gk[:, some].double().cpu()) <= 1e-5


def _backward_ws(w, k, g, B, C, T, ws, n):
    gw, gk = torch.full((C, T), 1e9, device=DEV), torch.full((B, C, T), 1e9, device=DEV)
    call("rwkv_timex_backward_ws", w.device, w, k, g, gw, gk, B, C, T, ws, n)
    return gw, gk


@pytest.mark.parametrize("B,C,T,parts", [(24, 600, 388, 0), (32, 768, 1500, 0), (13, 384, 1500, 2), (13, 64, 1500, 7)])
def test_a_workspace_for_fewer_groups(lib, B, C, T, parts):
    """What was enough when every lag tile had 32 lags (none at all for 512 channels and more) still is."""
    part = 4 * C * T
    assert lib.rwkv_timex_backward_ws_bytes(B, C, T) > max(parts, 1) * part
    some = [0, C // 2, C - 1]
    d, (_, gw, gk) = _some_channels(B, C, T, B + T, some)
    ws = torch.full((parts * C * T + 1024,), 7.5, device=DEV)
    got = _backward_ws(*d, B, C, T, ws if parts else None, parts * part)
    assert max_rel_to_peak(gw, got[0][some].double().cpu()) <= 1e-5 and max_rel_to_peak(gk, got[1][:, some].double().cpu()) <= 1e-5
    assert bool((ws[parts * C * T:] == 7.5).all())


@pytest.mark.parametrize("B,C,T,parts", [(13, 384, 1500, 2), (13, 64, 1500, 7), (30, 200, 300, 2)])
def test_a_workspace_for_too_few_groups_is_refused(lib, B, C, T, parts):
    d = [x.to(DEV) for x in synth.timex_inputs(B, C, T, seed=1)]
    ws = torch.empty(parts * C * T, device=DEV)
    for w, n in ((ws, 4 * parts * C * T - 4), (None, 0), (ws.data_ptr() + 4, 4 * parts * C * T)):
        with pytest.raises(RuntimeError):
            _backward_ws(*d, B, C, T, w, n)


def _rows_at_a_time(B, T, narrow):
    """How many batch rows a workgroup of the kernel gradient has in LDS at a time (gw_short_geom, gw_any_geom of timex.hip)."""
    nt, best = (T + 31) // 32, 1
    for bg in range(2, min(B, 32) + 1):
        if narrow:                      # three planes each of g and k in blocks of 40 elements, zero blocks between the rows, and the diagonals' sums
            zb = -(-15 // bg)
            zb += (nt + zb + 1) & 1
            size = 2 * 3 * (zb + bg * (nt + zb)) * 40 * 2 + 256 * nt + 16
        else:                           # three planes of g in blocks of 144 and of k; the eight waves' sums
            size = max(bg * 3 * (144 * ((nt + 3) // 4 + 1) + 32 * nt) * 2 + 16, 8 * 1024 * min(-(-T // 256), 8))
        if size > 80 * 1024 or 8 * nt * bg > 3 * 512:
            break
        best = bg
    return best


# B, T -> groups of rows that one workgroup takes one after the other, where the whole batch is its part (512 channels and more, no workspace)
GROUPS = {(13, 1500): 4, (9, 1500): 3, (13, 712): 2, (16, 1000): 4, (5, 2052): 3, (7, 4092): 7, (31, 516): 4, (33, 260): 3, (40, 384): 4, (64, 68): 2}


def _one_part(lib, B, T, monkey=None):
    """w, k, g of 512 channels, of which the rows of 0, 200 and 511 may be changed by `monkey`, and both sides' gradients of these."""
    C, some = 512, [0, 200, 511]
    at_a_time = _rows_at_a_time(B, T, T <= 384)
    assert -(-B // at_a_time) == GROUPS[B, T]
    w, k, g = synth.timex_inputs(B, C, T, seed=B + T)
    if monkey is not None:
        monkey(k, g)
    ref = OT.grads(w[some], k[:, some], g[:, some], B, 3, T)
    w, k, g = (x.to(DEV) for x in (w, k, g))
    gw, gk = _backward_ws(w, k, g, B, C, T, None, 0)
    return ref[1], gw[some].double().cpu(), ref[2], gk[:, some].double().cpu(), at_a_time


@pytest.mark.parametrize("B,T", list(GROUPS))
def test_groups_of_rows_one_after_the_other(lib, B, T):
    """Sums that are kept over groups, the next group's rows loaded under the products, a last group of fewer rows."""
    gw, got_gw, gk, got_gk, _ = _one_part(lib, B, T)
    assert max_rel_to_peak(gw, got_gw) <= 1e-5 and max_rel_to_peak(gk, got_gk) <= 1e-5


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 3.4e38])
@pytest.mark.parametrize("where", ["first", "middle", "first and last"])
@pytest.mark.parametrize("B,T", [(13, 1500), (9, 1500), (33, 260)])
def test_groups_with_an_element_that_terms_do_not_carry(lib, B, T, where, bad):
    """A group that is done by the fp32 loop before, between or after groups on the matrix cores: their sums add up, and lags that the
    element does not act on are finite.  3.4e38 is a number that three bf16 terms do not carry: nothing is lost."""
    rows = {"first": [1], "middle": [B // 2], "first and last": [0, B - 1]}[where]
    t0 = T - T // 3

    def put(k, g):
        g.clamp_(-0.9 / len(rows), 0.9 / len(rows))         # (the products add up to no more than fp32's largest)
        for i, b in enumerate(rows):
            k[b, 0, t0 + 2 * i] = bad

    gw, got, _, _, bg = _one_part(lib, B, T, put)
    groups = -(-B // bg)
    even = bg if T <= 384 else -(-B // groups)
    assert len({b // even for b in rows}) == len(rows) and (where != "middle" or 0 < rows[0] // even < groups - 1)
    lag = torch.arange(T - 1, -1, -1)
    hit = lag <= T - 1 - t0                                 # of channel 0
    if bad != 3.4e38:
        assert torch.equal(~torch.isfinite(got[0]), hit)
        assert max_rel_to_peak(gw[0][~hit], got[0][~hit]) <= 1e-5
    else:
        for z in (hit, ~hit):
            assert max_rel_to_peak(gw[0][z], got[0][z]) <= 1e-5
    assert max_rel_to_peak(gw[1:], got[1:]) <= 1e-5


def test_rows_of_very_different_size(lib):
    """The rows of a unit do not meet."""
    B, C, T = 6, 2, 500
    w, k, g = synth.timex_inputs(B, C, T, seed=4)
    scale = torch.tensor([1.0, 1e-4, 1e3, 1e-2, 1.0, 1e-3]).view(B, 1, 1)
    out, gw, gk = OT.grads(w, k * scale, g * scale, B, C, T)
    t = [x.to(DEV).requires_grad_(True) for x in (w, k * scale)]
    x = depthwise_conv1d.RUN_CUDA(*t, B, C, T, 0.0)
    x.backward((g * scale).to(DEV))
    for b in range(B):
        assert max_rel_to_peak(out[b], x[b].detach().double().cpu()) <= 1e-5 and max_rel_to_peak(gk[b], t[1].grad[b].double().cpu()) <= 1e-5, b


def _abs_sums(w, k, g, B, C, T):
    """What the fp32 bound is taken of, and how many products each sum has."""
    out, gw, gk = OT.grads(w.abs(), k.abs(), g.abs(), B, C, T)
    n = torch.arange(1, T + 1, dtype=torch.float64)
    return (out, n), (gw, B * n), (gk, n.flip(0))


@pytest.mark.parametrize("spike", [None, 1e6, 3.4e38])
@pytest.mark.parametrize("B,T", [(3, 4), (1, 36), (3, 60), (2, 500), (5, 1500), (2, 4096)])
def test_every_element_within_the_bound_of_an_fp32_loop(lib, B, T, spike):
    """Also in rows that are small until one large element (beyond bf16's range, too), which the elements before it do not see."""
    C = 2
    print(f"\ntimex any bound B={B} T={T} spike={spike}", flush=True)
    w, k, g = (x.clamp(-0.9, 0.9) for x in synth.timex_inputs(B, C, T, seed=3 * B + T))
    if spike is not None:
        m = T // 2
        k[:, :, :m] *= 1e-7
        k[0, :, m] = spike              # (in one row: its product with |w|, |g| <= 0.9 is below fp32's largest number, that of three rows is not)
        g[:, :, m + 1:] *= 1e-7
    ref = OT.grads(w, k, g, B, C, T)
    t = [x.to(DEV).requires_grad_(True) for x in (w, k)]
    x = depthwise_conv1d.RUN_CUDA(*t, B, C, T, 0.0)
    x.backward(g.to(DEV))
    for name, a, got, (mag, n) in zip(("x", "gw", "gk"), ref, (x, t[0].grad, t[1].grad), _abs_sums(w, k, g, B, C, T)):
        worst = ((got.detach().double().cpu() - a).abs() / ((n + 4) * 2.0 ** -24 * mag + 1e-38)).max().item()
        print(f"  {name}: worst element at {worst:.3f} of the bound", flush=True)
        assert worst <= 1, name


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("T", [60, 1500])
def test_an_element_that_is_no_number_stays_where_it_acts(lib, T, bad):
    """Not in other rows, in earlier outputs, or (mirrored) in later gradients."""
    B, C = 5, 2
    t0, t1 = T // 2 + 3, T // 3
    w, k, g = synth.timex_inputs(B, C, T, seed=T)
    kb, gb = k.clone(), g.clone()
    kb[1, 0, t0] = bad
    gb[3, 1, t1] = bad
    ref = OT.grads(w, k, g, B, C, T)
    t = [x.to(DEV).requires_grad_(True) for x in (w, kb)]
    x = depthwise_conv1d.RUN_CUDA(*t, B, C, T, 0.0)
    x.backward(gb.to(DEV))
    x, gw, gk = x.detach().double().cpu(), t[0].grad.double().cpu(), t[1].grad.double().cpu()
    hit_x = torch.zeros(B, C, T, dtype=torch.bool)
    hit_x[1, 0, t0:] = True
    hit_k = torch.zeros(B, C, T, dtype=torch.bool)
    hit_k[3, 1, :t1 + 1] = True
    lag = torch.arange(T - 1, -1, -1)
    hit_w = torch.stack([lag <= T - 1 - t0, lag <= t1])
    for name, a, got, hit in (("x", ref[0], x, hit_x), ("gw", ref[1], gw, hit_w), ("gk", ref[2], gk, hit_k)):
        assert torch.equal(~torch.isfinite(got), hit), name
        assert max_rel_to_peak(a[~hit], got[~hit]) <= 1e-5, name
