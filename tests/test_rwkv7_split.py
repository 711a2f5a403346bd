"""CPU: the split products of the chunked rwkv7 kernels (csrc/split3.h), restated in numpy.

An fp32 operand is three bf16 terms, x = h + m + l, each the nearest bf16 of the exact remainder, the first one never an
infinity; a product is the six of the nine that count.  Checked here: over which range the three terms hold all 24 bits, what
happens at its ends, and what the three products left out are worth."""
import os
import re

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rwkv_cuda_amd", "csrc")
FLT_MAX, BF_MAX = np.finfo(np.float32).max, np.float32((2 - 2.0 ** -7) * 2.0 ** 127)


def to_bf16(x):
    """Nearest bf16, ties to even, as fp32."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32)).view(np.float32)


def finite(h):
    """finite2 of split3.h: the same minima over 16-bit integers."""
    b = (h.view(np.uint32) >> 16).astype(np.uint16)
    b = np.minimum(b.view(np.int16), np.int16(0x7f7f)).view(np.uint16)
    b = np.minimum(b, np.uint16(0xff7f))
    return (b.astype(np.uint32) << 16).view(np.float32)


def split3(x):
    x = np.asarray(x, np.float32)
    h = finite(to_bf16(x))
    r = x - h
    m = to_bf16(r)
    return h, m, to_bf16(r - m)


def values(lo, hi, n=200000, seed=0):
    """Magnitudes spread over the logarithm, random significands and signs."""
    rng = np.random.default_rng(seed)
    x = np.ldexp(rng.uniform(1, 2, n), rng.integers(lo, hi, n)).astype(np.float32)
    return x * rng.choice(np.float32([-1, 1]), n)


def test_three_terms_hold_all_24_bits():
    x = values(-110, 128)
    x = np.concatenate([x, np.float32([FLT_MAX, -FLT_MAX, BF_MAX, -BF_MAX, 2.0 ** -110, 0.0])])
    edge = np.arange(0x7f7f0000, 0x7f800000, dtype=np.uint32).view(np.float32)          # around and beyond the largest bf16
    for v in (x, edge, -edge):
        h, m, l = split3(v)
        assert np.all(np.isfinite(h)) and np.all(np.isfinite(m)) and np.all(np.isfinite(l))
        assert np.array_equal(h.astype(np.float64) + m + l, v.astype(np.float64))


def test_the_first_term_is_the_nearest_bf16_up_to_the_largest():
    x = values(-126, 128)
    x = x[np.abs(x) <= BF_MAX]
    assert np.array_equal(split3(x)[0], to_bf16(x))
    assert np.array_equal(split3(np.float32([FLT_MAX, -FLT_MAX]))[0], np.float32([BF_MAX, -BF_MAX]))


def test_smaller_values_lose_bits_to_the_spacing_of_bf16_subnormals():
    x = values(-126, -110)
    h, m, l = split3(x)
    err = np.abs(h.astype(np.float64) + m + l - x.astype(np.float64))
    assert err.max() <= 2.0 ** -134 and err.max() > 0          # half of 2^-133


@pytest.mark.parametrize("v", [np.inf, -np.inf, np.nan])
def test_an_infinity_or_nan_is_not_finite_in_its_remainders(v):
    with np.errstate(invalid="ignore"):
        h, m, l = split3(np.float32([v]))
        assert np.isnan((h.astype(np.float64) + m + l)[0])


def test_products_left_out():
    """m l' + l m' + l l' against the whole product: at most 2^-24, 2^-27 in the root mean square."""
    x, y = values(-1, 1, seed=1), values(-1, 1, seed=2)
    (h, m, l), (p, q, s) = ([t.astype(np.float64) for t in split3(v)] for v in (x, y))
    exact = x.astype(np.float64) * y
    six = h * p + h * q + m * p + m * q + h * s + l * p
    rel = np.abs(six - exact) / np.abs(exact)
    assert rel.max() <= 2.0 ** -24 and np.sqrt((rel ** 2).mean()) <= 2.0 ** -27


@pytest.mark.parametrize("name", ["split3.h", "rwkv7_chunk.hip"])
def test_no_instruction_is_inline_assembly(name):
    """Operands of matrix instructions are made here.  Such an instruction needs two wait states after the vector instruction that writes
    its operand; the compiler inserts them, but not for an instruction inside assembly.  Empty asm statements (values kept from the
    optimiser) are no instruction."""
    with open(os.path.join(CSRC, name)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    bodies = re.findall(r"\basm\b(?:\s+volatile)?\s*\(\s*\"([^\"]*)\"", text)
    assert bodies and all(b == "" for b in bodies), bodies


def decay_parts(sig):
    """decay_of_sig of csrc/rwkv7_chunk.hip, fused operations in fp64 and rounded (HI, LO: the two constants)."""
    f = np.float32
    C = -0.6065306597 * 1.4426950408889634
    HI = f(C)
    LO = f(C - float(HI))
    fma = lambda a, b, c: (a.astype(np.float64) * np.float64(b) + c).astype(f)
    hi = fma(sig, HI, 24.0) - f(24)
    return hi, (f(0.69314718055994530942) * fma(sig, LO, fma(sig, HI, -hi.astype(np.float64)).astype(np.float64))).astype(f)


def test_decays_of_a_chunk_add_up_exactly():
    """Sums of the first parts over 16 steps are exact in any order, the second parts stay below 2^-20, and e to the sum of both is off by
    the exponential's rounding and a few of 2^-40: 1e-7 where a sum of fp32 decays is off by 4e-7."""
    rng = np.random.default_rng(3)
    sig = np.concatenate([rng.uniform(0, 1, (4000, 16)), 1 / (1 + np.exp(rng.uniform(0, 12, (4000, 16)))), np.ones((1, 16)), np.zeros((1, 16))]).astype(np.float32)
    hi, lo = decay_parts(sig)
    assert np.all(np.abs(lo) <= 2.0 ** -20)
    for order in (slice(None), slice(None, None, -1)):
        run = np.cumsum(hi[:, order], axis=1, dtype=np.float32)
        assert np.array_equal(run.astype(np.float64), np.cumsum(hi[:, order].astype(np.float64), axis=1))
    total = lo[:, 0].copy()
    for t in range(1, 16):
        total += lo[:, t]
    got = np.exp2(hi.astype(np.float64).sum(1)).astype(np.float32)
    got = (got.astype(np.float64) * total + got).astype(np.float32).astype(np.float64)
    want = np.exp(-0.6065306597 * sig.astype(np.float64).sum(1))
    assert np.max(np.abs(got / want - 1)) <= 2 * 2.0 ** -24 + 2.0 ** -32


def test_constants_of_the_decay():
    """The quotient of the two constants of decay_of is W_SCALE log2(e) to 1e-12, where the nearest fp32 number is 3e-8 off."""
    with open(os.path.join(CSRC, "rwkv7_chunk.hip")) as f:
        m = re.search(r"constexpr float C = (0x[0-9a-f.p+-]+)f, M = (-0x[0-9a-f.p+-]+)f;", f.read())
    C, M = (float.fromhex(z) for z in m.groups())
    assert float(np.float32(C)) == C and float(np.float32(M)) == M
    assert abs(M / C / (-0.6065306597 * 1.4426950408889634) - 1) < 1e-12


def decay_sources():
    """The two forms of a step's decay in csrc/rwkv7_chunk.hip, from a sigmoid (backward) and from the input (forward, blocks), with the source's
    own constants: functions of the input in fp64 that give the two parts, fused operations in fp64 and rounded."""
    with open(os.path.join(CSRC, "rwkv7_chunk.hip")) as f:
        text = f.read()
    f32, fma = np.float32, lambda a, b, c: (a.astype(np.float64) * np.float64(b) + c).astype(np.float32)
    ln2 = f32(float(re.search(r"constexpr float LN2 = ([\d.]+)f;", text).group(1)))
    a = text[text.index("DEVINL Decay decay_of_sig(float sig) {"):]
    a = a[:a.index("\n}")]
    w, log2e = map(float, re.search(r"constexpr double C = (-[\d.]+) \* ([\d.]+);", a).groups())
    assert "HI = static_cast<float>(C), LO = static_cast<float>(C - static_cast<double>(HI));" in a
    off = {float(z) for z in re.search(r"hi = fmaf\(sig, HI, ([\d.]+)f\) - ([\d.]+)f;", a).groups()}
    assert "return {hi, LN2 * fmaf(sig, LO, fmaf(sig, HI, -hi))};" in a
    HI = f32(w * log2e)
    LO = f32(w * log2e - float(HI))
    b = text[text.index("DEVINL Decay decay_of(float x) {"):]
    b = b[:b.index("\n}")]
    C, M = (float.fromhex(z) for z in re.search(r"constexpr float C = (\S+)f, M = (\S+)f;", b).groups())
    assert "d = fmaf(__builtin_amdgcn_exp2f(x * -1.44269504088896340736f), C, C);" in b and "return {hi, LN2 * fmaf(s, M, -hi)};" in b
    off |= {float(z) for z in re.search(r"hi = fmaf\(s, M, ([\d.]+)f\) - ([\d.]+)f;", b).groups()}
    assert len(off) == 1
    off = off.pop()

    def of_sig(x):
        sig = (1 / (1 + np.exp(-x))).astype(f32)
        hi = fma(sig, HI, off) - f32(off)
        return hi, ln2 * fma(sig, LO, fma(sig, HI, -hi.astype(np.float64)).astype(np.float64))

    def of_input(x):
        s = (1 / (C * (1 + np.exp(-x)))).astype(f32)
        hi = fma(s, M, off) - f32(off)
        return hi, ln2 * fma(s, M, -hi.astype(np.float64))

    return of_sig, of_input


def test_both_forms_of_the_decay_add_up_exactly_and_agree():
    """The backward uses states that the forward has decayed.  Bound of their difference: a sigmoid's rounding of 2^-24 and a product's of 2^-24
    each, of the sum of 16; second parts to 2^-24 of 2^-20."""
    rng = np.random.default_rng(4)
    x = np.concatenate([rng.normal(c, s, (2000, 16)) for c in (-8, -5, -2, 0.5, 3) for s in (0, 1)] + [np.full((1, 16), z) for z in (30.0, 0.0, -80.0)])
    exact = -0.6065306597 / (1 + np.exp(-x))
    totals = []
    for form in decay_sources():
        hi, lo = form(x)
        assert np.all(np.abs(lo) <= 2.0 ** -20) and np.all(np.abs(hi) < 1) and np.all(hi * 2.0 ** 19 == np.round(hi * 2.0 ** 19))
        for order in (slice(None), slice(None, None, -1), rng.permutation(16)):
            assert np.array_equal(np.cumsum(hi[:, order], axis=1, dtype=np.float32), np.cumsum(hi[:, order].astype(np.float64), axis=1))
        totals.append(hi.astype(np.float64).sum(1) * np.log(2) + lo.astype(np.float64).sum(1))
        assert np.all(np.abs(totals[-1] - exact.sum(1)) <= np.abs(exact).sum(1) * 2.0 ** -23 + 16 * 2.0 ** -44)
    assert np.all(np.abs(totals[0] - totals[1]) <= np.abs(exact).sum(1) * 2.0 ** -22 + 32 * 2.0 ** -44)
