// RWKV-7 "clamp-w" generalised delta rule in CHUNKED form on the matrix cores (gfx950).
//
// Step form (rwkv7_fast_fused/cuda/rwkv7_statepassing_clampw.cu:20-187), one head, S[i][j] (i value, j key):
//     sa_t = S_t a_t;   S_{t+1} = S_t diag(w_t) + sa_t b_t^T + v_t k_t^T;   y_t = S_{t+1} r_t;   w_t = exp(W_SCALE sigmoid(w_raw_t))
// A chunk of L = 16 steps (the reference's CHUNK_LEN), local t = 0..15, S0 the state entering it, lam_t = log w_t, c_t = sum_{z<t} lam_z.
// Everything is referred to one border of the chunk, e^{+-9.8} at most, so nothing needs a fallback.  Forward, to the chunk's end, with
// x_t = e^{c_L - c_t}, dec = x_0 = e^{c_L}:
//     A_t = a_t / x_t    R_t = r_t / x_{t+1}    B_s = b_s x_{s+1}    K_s = k_s x_{s+1}    D0 = S0 diag(dec)
//     AB = tril_-(A B^T)  AK = tril_-(A K^T)  RB = tril(R B^T)  RK = tril(R K^T)                         [16 x 16]
//     U  = (I - AB)^{-1} (A D0^T + AK V)               rows of U are sa_t (the tensor `sa` of the interface)
//     Y  = R D0^T + RB U + RK V
//     S_L = D0 + U^T B + V^T K
// So each input is multiplied and split once: A and R meet the state and make the tiles, B and K make the tiles and the new state.  What
// is near the end, the largest part of that, has the smallest exponents.  (Referred to the middle for the tiles, to the start for A and R and to
// the end for B and K, which is as accurate, the four inputs were eight planes.)
// Backward of a chunk from dY and dS_L (the gradient w.r.t. S_L through everything after the chunk), referred to the chunk's start, with
// x_t = e^{c_t}, dec = x_L, A_t = a_t x_t, R_t = r_t x_{t+1}, B_s = b_s / x_{s+1}, K_s = k_s / x_{s+1}, E = dS_L diag(dec) (the tiles are the same):
//     dU  = RB^T dY + B E^T                   dW = (I - AB)^{-T} dU
//     dAB = tril_-(dW U^T)  dAK = tril_-(dW V^T)  dRB = tril(dY U^T)  dRK = tril(dY V^T)
//     dV  = AK^T dW + RK^T dY + K E^T
//     dS0 = E + dY^T R + dW^T A
//     dA = dAB B + dAK K + dW S0              dR = dRB B + dRK K + dY S0
//     dB = dAB^T A + dRB^T R + U E            dK = dAK^T A + dRK^T R + V E
//     da = dA x_t, dr = dR x_{t+1}, db = dB / x_{t+1}, dk = dK / x_{t+1}
//     decay: with P_t = sum_i dS_t o S_t per key channel,  G_t = P_{t+1} + r dr - b db - k dk,  P_t = G_t + a da,
//            dw_raw = G W_SCALE sig (1 - sig);  P at the end of the call = sum_i dsT o S_T.
// What is divided by x is held by 2^-7 (HOLD below).
// Every product takes all 24 bits of its operands, so the fp32 outputs sT, ds0 and the saved sa keep the accuracy class of the
// reference's fp32 recurrence; the bf16 outputs are rounded once at the store.  The fp32 mode is therefore the same kernel with fp32
// loads and stores.  Products are split ones (split3.h); the few of the scan over blocks are fp32 matrix instructions.
//
// One workgroup per (batch, head).  A 16x16 matrix instruction leaves D[row = 4 (lane >> 4) + v][col = lane & 15] in register v.  The state is
// kept TRANSPOSED in accumulator registers, S^T tile jt of wave q: register v of lane (l16, g) = S[i = 16 q + l16][j = 16 jt + 4 g + v].
// K slots may be assigned to channels (or tokens) in any order as long as both operands agree, so accumulator registers, split, are the
// B operand of the next product: two state tiles of a contraction over 32 channels, U, W, dU, dW of one over 16 tokens.  Nothing is
// transposed through LDS but by reads that transpose.
//
// Private layout of the interface's scratch tensors: `s` slot c holds the state ENTERING chunk c as [i][j] fp32 (the
// reference stores the state leaving it; the backward here needs the entering one and never inverts a step), `sa` is U.
#include <stddef.h>
#include <algorithm>

#include "split3.h"

namespace rwkv {
namespace {

constexpr int N = 64;
constexpr int CL = RWKV7_CHUNK_LEN;
constexpr int PS = 68;            // row stride (floats) of a [token][channel] plane
constexpr int TS = 20;            // row stride (floats) of a 16 x 16 tile
constexpr float W_SCALE = -0.6065306597f;   // -exp(-0.5), rwkv7_statepassing_clampw.cu:16

DEVINL f32x4 mm(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
DEVINL f32x4 ld4(const float* p) { const float4 x = *reinterpret_cast<const float4*>(p); return f32x4{x.x, x.y, x.z, x.w}; }
DEVINL void st4(float* p, const f32x4& x) { *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]); }
// What only a backward reads again, 20 bytes an element: marked not to stay in the caches, where it would take the place of the rows that are
// coming in.  B=1, T=4096, H=32, forward that keeps its states: bf16 185 -> 178 us, fp32 211 -> 198; B=8, T=1024, H=64: 336 -> 333 and
// 369 -> 365.  Not so for what the forward returns (fp32 365 -> 377), nor for the backward's reads of the states (fp32 638 -> 655).
DEVINL void st4_stream(float* p, const f32x4& x) { __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(p)); }
constexpr f32x4 ZERO4 = {0.f, 0.f, 0.f, 0.f};

// Element pointers are typed for the bf16 mode; the fp32 mode (the reference's -D_FP32_ build) keeps float pointers in the
// same fields and its instantiations (F32 = true) read and write them as such.
struct Args7c {
    int T, H;
    const uint16_t *r, *w, *k, *v, *a, *b, *dy;
    const float *s0, *dsT;
    uint16_t *y, *dr, *dw, *dk, *dv, *da, *db;
    float *sT, *ds0;
    float* s;     // [B,H,T/16][i][j]: state entering each chunk
    float* sa;    // [B,T,H,N]: U
    // sequences cut into NB > 1 blocks of `per` chunks, a workgroup each (blockIdx.z); per head: what each block makes of a state (local:
    // E and M of the blocks but the last in the direction of travel), the states entering the blocks but the first (enter), whether the
    // head is done as a whole (flags)
    int NB, per;
    int at;       // this launch's first head, batch row by batch row (local, enter and flags begin with it)
    float *local, *enter;
    int* flags;
};

// Whole sequences (CUT = false) have an instance of their kernels of their own: with the choice left to run time what belongs to the
// blocks costs them scalar work (B8 4 x T1024 C4096 3.87 -> 3.83 ms).
template <bool CUT> DEVINL Args7c only_whole(Args7c p) {
    if constexpr (!CUT) p.NB = 1;
    return p;
}
// head n of the launch
struct Head7 { size_t bh; int b, h; };
DEVINL Head7 head_of(const Args7c& p, int n) {
    const int bh = p.at + n, b = __builtin_amdgcn_readfirstlane(bh / p.H);
    return {static_cast<size_t>(bh), b, bh - b * p.H};
}
// The state of head bh (s0 or dsT) that the first block in the direction of travel starts from.  In blocks it is the copy that rwkv7c_scan leaves
// in the place of the first block's E: the last block may have written sT (ds0) by then, and that may be the same tensor.
DEVINL const float* first_state(const Args7c& p, const float* x, size_t bh) {
    if (x == nullptr) return nullptr;
    return p.NB > 1 ? p.local + static_cast<size_t>(blockIdx.x) * (p.NB - 1) * 2 * N * N : x + bh * N * N;
}
// The chunks of the workgroup's block; false: another workgroup does them.
struct Part7 { int n, first, chunks; };
DEVINL bool part_of(const Args7c& p, Part7& x) {
    const int nch = p.T / CL;
    x = {0, 0, nch};
    if (p.NB == 1) return true;
    if (__builtin_amdgcn_readfirstlane(p.flags[blockIdx.x]) != 0) return blockIdx.z == 0;
    x.n = blockIdx.z; x.first = x.n * p.per; x.chunks = min(p.per, nch - x.first);
    return true;
}

// element base + o as it comes from memory, and its value
// (a scalar base and one 32-bit byte offset a lane)
template <bool F32> DEVINL uint32_t ld_raw(const uint16_t* p, size_t base, uint32_t o) {
    const char* const b = reinterpret_cast<const char*>(p) + base * (F32 ? 4 : 2);
    if constexpr (F32) return *reinterpret_cast<const uint32_t*>(b + o * 4u);
    else return *reinterpret_cast<const uint16_t*>(b + o * 2u);
}
template <bool F32> DEVINL float widen(uint32_t x) { return F32 ? __uint_as_float(x) : bf2f(static_cast<uint16_t>(x)); }

// the four values x[4 g + v] of lane group g (behind an empty asm: the compiler would make branches of the choice, with the sums in them)
DEVINL f32x4 by_group(int g, float (&x)[CL]) {
#pragma unroll
    for (int i = 0; i < CL; ++i) asm volatile("" : "+v"(x[i]));
    f32x4 r;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float lo = g & 1 ? x[4 + v] : x[v], hi = g & 1 ? x[12 + v] : x[8 + v];
        r[v] = g & 2 ? hi : lo;
    }
    return r;
}

// M = (I - AB)^{-1}, four copies in the four rows of lanes.  The lane that holds line n of the triangle gives the others the element that they
// need inside the multiplication, so the tile is read once.  (With every element read from LDS where it was needed, 38 reads in a chain, the
// wave that makes M took 5100 cycles of the forward's phase and the others 3400: B=8, T=1024, H=64 without a gradient 243 -> 240 us in bf16 and
// 283 -> 274 in fp32, fp32 backward 642 -> 631; B=1, T=4096, H=32 without a gradient 175 -> 164 and 183 -> 175.)
// ROWS: lane l16 = r gets M[r][0 .. 15] from M[r][s] = [r == s] + sum_{t>s} M[r][t] AB[t][s]; lines holds AB[.][s] as its row s.
// Otherwise lane l16 = c gets M[0 .. 15][c] from M[t][c] = [t == c] + sum_{s<t} AB[t][s] M[s][c]; lines holds AB itself.
template <bool ROWS> DEVINL void inverse(const float (*lines)[TS], int l16, float (&m)[CL]) {
    float x[CL];
#pragma unroll
    for (int i = 0; i < CL; i += 4) {
        const f32x4 y = ld4(&lines[l16][i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[i + e] = y[e];
    }
    asm volatile("" : "+v"(l16));            // (or sixteen comparisons with it live in registers across the caller's loop)
#pragma unroll
    for (int i = 0; i < CL; ++i) m[i] = l16 == i ? 1.f : 0.f;
    solve_bc<ROWS>(m, x);
}

// (a Newton step behind the hardware reciprocal instead of a full division, a sixth of the vector instructions that turn inputs into
// planes.  A quarter of the denominator, since the reciprocal flushes what is below 2^-126; an overflown exponential leaves zero, and
// so no decay gradient, where the step by itself would make a NaN; a NaN passes by y)
DEVINL float sigmoid_fast(float x) {
    const float d = fmaf(__builtin_amdgcn_exp2f(x * -1.44269504088896340736f), 0.25f, 0.25f);
    const float y = __builtin_amdgcn_rcpf(d);
    return 0.25f * fmaf(fmaf(-fminf(d, 3.40282346638528859812e38f), y, 1.f), y, y);
}

// Decay of a step in two parts, in units of log 2 a multiple of 2^-19 below 1, of which sums over a chunk (below 14) are exact, and in those
// of e the rest, below 2^-20: with the sum of the first parts rounded to fp32 an exponential is off by up to 3e-7.
struct Decay { float hi, lo; };
constexpr float LN2 = 0.69314718055994530942f;
DEVINL Decay add(const Decay& a, const Decay& b) { return {a.hi + b.hi, a.lo + b.lo}; }
// e to a sum of decays: the hardware's exponential of the nearest exponent; what that leaves is mostly below half a place of the result, so
// that it is rounded once.  (exp2 of the first part times 1 + lo is rounded twice: at w = -3 to -8 that is 3 % of the errors of what a
// chunk hands on and of dv, dk.)
DEVINL float grow(const Decay& d) {
    const float t = fmaf(d.lo, 1.44269504088896340736f, d.hi), rest = fmaf(LN2, d.hi - t, d.lo), e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, rest, e);
}
// W_SCALE log2(e) sigmoid(x), from the sigmoid
DEVINL Decay decay_of_sig(float sig) {
    constexpr double C = -0.6065306597 * 1.44269504088896340736;
    constexpr float HI = static_cast<float>(C), LO = static_cast<float>(C - static_cast<double>(HI));
    const float hi = fmaf(sig, HI, 24.f) - 24.f;                   // (24: whose last place is 2^-19)
    return {hi, LN2 * fmaf(sig, LO, fmaf(sig, HI, -hi))};
}
// The factors of the four tokens (4 q + e) of a channel held by a thread, from their decays (part: the waves' sums of them).  All four
// inputs are referred to one border of the chunk, forwards its end, backwards its start, so that each is split once and
// serves both the causal tiles and the state: x[e] = e^{c_L - c_t} (e^{c_t}), t = 4 q + e, e = 0 .. 4, carry to or from the border what
// is added to the state that is handed on, y[e] = HOLD / x[e] meet the state that came in, which has the chunk's whole decay on it
// beforehand.  HOLD: or e^9.7 would take inputs out of range that e^4.9 (referred to the chunk's middle) did not.
// (NEAREST: with a Newton step, which the fp32 results of a backward show and bf16 ones do not)
constexpr float HOLD = 0.0078125f, UNHOLD = 128.f;
template <bool NEAREST> DEVINL float held_inverse(float x) {
    float y = __builtin_amdgcn_rcpf(x);
    if constexpr (NEAREST) y = fmaf(fmaf(-x, y, 1.f), y, y);
    return y * HOLD;
}
template <bool END, bool NEAREST> DEVINL void growth(const Decay (&lam)[4], const Decay (*part)[N], int q, int j, float (&x)[5], float (&y)[5]) {
    Decay at = {0.f, 0.f};                             // between the thread's tokens and the border
    const int n = END ? 3 - q : q, d = END ? -1 : 1, b = END ? 3 : 0;
    if (n > 0) at = part[b][j];
    if (n > 1) at = add(at, part[b + d][j]);
    if (n > 2) at = add(at, part[b + 2 * d][j]);
#pragma unroll
    for (int z = 0; z < 5; ++z) {
        const int e = END ? 4 - z : z;
        if (z > 0) at = add(at, lam[END ? e : e - 1]);
        x[e] = grow(at);
        y[e] = held_inverse<NEAREST>(x[e]);
    }
}
// e to the chunk's whole decay, within half a place: the state takes it on in every chunk, and where it decays slowly its error adds up (64
// chunks of w = -8: sT 1.10e-7 off with the hardware's exponential, 1.25 with its remainder multiplied in, 1.07 so).  A power of two and
// the series of e^t for |t| < 0.35, to t^7.  (One coefficient behind an empty asm, or it takes a register across the loop.)
DEVINL float whole_decay(const Decay (*part)[N], int j) {
    const Decay d = add(add(part[0][j], part[1][j]), add(part[2][j], part[3][j]));
    const float n = __builtin_rintf(d.hi), t = fmaf(d.hi - n, LN2, d.lo);
    float p = 1.f / 5040;
    asm volatile("" : "+v"(p));
    p = fmaf(t, p, 1.f / 720); p = fmaf(t, p, 1.f / 120); p = fmaf(t, p, 1.f / 24); p = fmaf(t, p, 1.f / 6); p = fmaf(t, p, 0.5f);
    return __builtin_ldexpf(1.f + fmaf(t * t, p, t), static_cast<int>(fmaxf(n, -16.f)));            // (fmaxf: a NaN is no integer)
}
DEVINL Decay sum4(const Decay (&l)[4]) { return add(add(l[0], l[1]), add(l[2], l[3])); }
// the same from x, in a backward-less chain: c / (1 + e^-x) with the quotient of the two constants 3e-13 from the product
DEVINL Decay decay_of(float x) {
    constexpr float C = 0x1.fee3f2p-3f, M = -0x1.bf0c86p-3f;
    const float d = fmaf(__builtin_amdgcn_exp2f(x * -1.44269504088896340736f), C, C);
    const float y = __builtin_amdgcn_rcpf(d), s = fmaf(fmaf(-fminf(d, 3.40282346638528859812e38f), y, 1.f), y, y);
    const float hi = fmaf(s, M, 24.f) - 24.f;
    return {hi, LN2 * fmaf(s, M, -hi)};
}

// HOLD tile[t][s] = sum_c a_t e^{c_t} b_s e^{-c_{s+1}} over 64 channels, masked to s < t (strict) or s <= t: register v <-> t = 4 g + v, lane <-> s,
// or (ROWS) register v <-> s = 4 g + v, lane <-> t.  ta, sb: operand of 32 channels of the t side, of the s side.
template <bool ROWS, class TA, class SB> DEVINL f32x4 causal_tile(TA ta, SB sb, bool strict, int l16, int g) {
    Sum2 sum = SUM0;
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
        const Op3 x = ta(hb), y = sb(hb);
        if constexpr (ROWS) add32(sum, y, x); else add32(sum, x, y);
    }
    f32x4 acc = total(sum);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int t = ROWS ? l16 : 4 * g + v, s = ROWS ? 4 * g + v : l16;
        acc[v] = (strict ? s < t : s <= t) ? acc[v] : 0.f;
    }
    return acc;
}

// ---------------------------------------------------------------------------------------------------- forward
// One workgroup of eight waves per (batch, head), two of them on a CU, two roles with their own loops and two barriers a chunk:
//          phase X                                                   | phase Y
//   S:     A D0^T, R D0^T; rows of the chunk before and the state     | AK V, U, RK V + RB U, the state
//          entering to memory                                         |
//   P:     causal tiles and the inverse of this chunk; decay sums of  | factors, planes of the next chunk
//          the next                                                   |
// A plane that one phase writes and the other reads needs no second copy (B, K and dec, which S reads while P writes, do).
constexpr int NTF = 8 * 64;        // waves 0..3 role S, 4..7 role P
struct SmemCF {
    float Yo[CL][PS], Uo[CL][PS];
    float ABt[CL][TS];
    Decay part[4][N];
    float dec[2][N];
};
// three-term planes and tiles behind it: HOLD A, HOLD R, K and B, v (one term where it is bf16), AK, RB, RK, (I - AB)^{-1}
constexpr uint32_t F_AS = (sizeof(SmemCF) + 31) / 32 * 32, F_RS = F_AS + PLANE3, F_KB = F_RS + PLANE3, F_V = F_KB + 2 * TWIN3;
template <bool F32> constexpr uint32_t F_MA = F_V + (F32 ? PLANE3 : TERM);      // (I - AB)^{-1} and AK
template <bool F32> constexpr uint32_t F_RKB = F_MA<F32> + TPAIR3;                // RK and RB
template <bool F32> constexpr uint32_t F_TOTAL = F_RKB<F32> + TPAIR3;
static_assert(F_TOTAL<true> <= 80 * 1024, "two workgroups a CU");

template <bool F32> DEVINL void fwd_role_p(SmemCF& S, const lds_t sb, const Args7c& p, int q, int lane, size_t tok0, int nch, int h) {
    const int l16 = lane & 15, g = lane >> 4, H = p.H;
    // channel j = lane, tokens 4 q + e
    uint32_t nx[6][4];
    auto fetch = [&](int c) __attribute__((always_inline)) {         // (clamped, so that every chunk issues the same loads)
        const size_t base = ((tok0 + static_cast<size_t>(c < nch ? c : nch - 1) * CL) * H + h) * N;
        uint32_t lo = lane;
        asm volatile("" : "+v"(lo));
        const uint16_t* const src[6] = {p.w, p.r, p.k, p.v, p.a, p.b};
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int k = 0; k < 6; ++k) nx[k][e] = ld_raw<F32>(src[k], base, static_cast<uint32_t>((4 * q + e) * H) * N + lo);
    };
    Decay lam[4];
    float rr[4], kk[4], aa[4], bb[4];
    [[maybe_unused]] float vv[4];
    [[maybe_unused]] uint32_t vb[4];
    auto convert = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            lam[e] = decay_of(widen<F32>(nx[0][e]));
            // (a value of its own: the product could join an addition in one of the two copies of this code and not in the other, and a
            // sequence cut into calls would no longer give the same bits)
            asm volatile("" : "+v"(lam[e].hi), "+v"(lam[e].lo));
            rr[e] = widen<F32>(nx[1][e]); kk[e] = widen<F32>(nx[2][e]);
            if constexpr (F32) vv[e] = widen<F32>(nx[3][e]); else vb[e] = nx[3][e];
            aa[e] = widen<F32>(nx[4][e]); bb[e] = widen<F32>(nx[5][e]);
        }
        S.part[q][lane] = sum4(lam);
    };
    auto planes = [&](const int slot) __attribute__((always_inline)) {
        float x[5], y[5];
        growth<true, false>(lam, S.part, q, lane, x, y);
        f32x4 as, rs, ks, bs;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            as[e] = aa[e] * y[e];
            rs[e] = rr[e] * y[e + 1];
            ks[e] = kk[e] * x[e + 1];
            bs[e] = bb[e] * x[e + 1];
        }
        const lds_t o = sb + piece(lane, q);
        put3(o + F_AS, split3(as)); put3(o + F_RS, split3(rs));
        // (x is not above 1: what comes from bf16 inputs stays within bf16's range)
        put_twin(sb + F_KB + slot * TWIN3 + twin(lane, q), split3<!F32>(ks), split3<!F32>(bs));
        if constexpr (F32) put3(o + F_V, split3(f32x4{vv[0], vv[1], vv[2], vv[3]}));
        else lds_st<u32x2>(o + F_V, u32x2{vb[0] | (vb[1] << 16), vb[2] | (vb[3] << 16)});
        if (q == 0) S.dec[slot][lane] = whole_decay(S.part, lane);
    };
    const Tr ta = tr_bases(sb + (q < 2 ? F_AS : F_RS), l16, g);
    const lds_t sp = tr_twin(sb + F_KB + ((q & 1) ? 0 : 32), l16, g);
    fetch(0);
    convert();
    fetch(1);
    __syncthreads();
    planes(0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        // ---------------------------------------------------------------- phase X
        {
            f32x4 x;
            auto top = [&](int hb) __attribute__((always_inline)) { return get3_tr(0, ta, hb); };
            auto sop = [&](int hb) __attribute__((always_inline)) { return get3_tr_twin(0, sp + (c & 1) * TWIN3, hb); };
            if (q == 0) {
                st4(&S.ABt[l16][4 * g], causal_tile<false>(top, sop, true, l16, g) * UNHOLD);
                // this wave wrote AB itself (LDS keeps a wave's accesses in order): the inverse once, for all four S waves
                float m[CL];
                inverse<true>(S.ABt, l16, m);
                x = by_group(g, m);
            } else x = causal_tile<true>(top, sop, q == 1, l16, g);
            // (one store with a selected address, as in the backward)
            put_half<TTERM2>(sb + piece2(l16, g) + (q == 0 ? F_MA<F32> : (q == 1 ? F_MA<F32> + 8 : (q == 2 ? F_RKB<F32> + 8 : F_RKB<F32>))), split3(x));
        }
        convert();
        fetch(c + 2);
        __syncthreads();
        // ---------------------------------------------------------------- phase Y
        planes((c + 1) & 1);
        __syncthreads();
    }
}

// s0, sT, slots: of this head and block
template <bool F32, bool KEEP> DEVINL void fwd_role_s(SmemCF& S, const lds_t sb, const Args7c& p, const float* s0, float* sT, float* slots, int q, int tid, size_t tok0, int nch, int h) {
    const int lane = tid & 63, l16 = lane & 15, g = lane >> 4, H = p.H;
    const int i_own = 16 * q + l16;
    // state, transposed tiles: St[jt][v] = S[i_own][16 jt + 4 g + v]
    f32x4 St[4];
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
        St[jt] = s0 != nullptr ? ld4(s0 + static_cast<size_t>(i_own) * N + 16 * jt + 4 * g) : ZERO4;
    // y and sa = U (fp32) of chunk c as whole rows
    auto store_rows = [&](const int c) __attribute__((always_inline)) {
        const int t = tid >> 4, i4 = (tid & 15) * 4;
        const size_t o = ((tok0 + static_cast<size_t>(c) * CL + t) * H + h) * N + i4;
        const f32x4 y = ld4(&S.Yo[t][i4]);
        if constexpr (F32) st4(reinterpret_cast<float*>(p.y) + o, y);
        else *reinterpret_cast<uint2*>(p.y + o) = make_uint2(pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]));
        if constexpr (KEEP) st4_stream(p.sa + o, ld4(&S.Uo[t][i4]));
    };
    const Tr tr = tr_bases(sb, l16, g);
    const lds_t pp = sb + piece2(l16, g), vp = sb + F_V + piece(i_own, g), kbs = sb + F_KB + twin(l16, g);
    auto load_v = [&]() __attribute__((always_inline)) {
        if constexpr (F32) return get3(vp); else return lds_ld<u32x2>(vp);
    };
    __syncthreads();
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        // ---------------------------------------------------------------- phase X: what needs no tile
        const auto vop = load_v();                   // V[s = 4 g + v][i_own]
        const float* const dec = &S.dec[c & 1][4 * g];
        Sum2 W = SUM0, Y = SUM0;                     // HOLD W, HOLD Y
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            // (decayed for these products only: in the update a fused multiplication and addition rounds the state once)
            const Op3 st = join(split3(St[2 * hb] * ld4(dec + 32 * hb)), split3(St[2 * hb + 1] * ld4(dec + 32 * hb + 16)));
            add32(W, get3_tr(F_AS, tr, hb), st);
            add32(Y, get3_tr(F_RS, tr, hb), st);
        }
        here(W); here(Y);
        if (c > 0) store_rows(c - 1);
        // the state entering the chunk, for the backward
        if constexpr (KEEP) {
            float* slot = slots + static_cast<size_t>(c) * N * N + static_cast<size_t>(i_own) * N + 4 * g;
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) st4_stream(slot + 16 * jt, St[jt]);
        }
        __syncthreads();
        // ---------------------------------------------------------------- phase Y
        add16(W, get_half<TTERM2>(pp + F_MA<F32> + 8), vop);
        Sum2 Us = SUM0;
        add16(Us, get_half<TTERM2>(pp + F_MA<F32>), split3(total(W) * UNHOLD));
        const f32x4 U = total(Us);
        const Op3 vu = join(as3(vop), split3(U));        // V and U share the instructions of what follows
        add32(Y, get_pair<TTERM2>(pp + F_RKB<F32>), vu);
        const f32x4 y = total(Y) * UNHOLD;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            S.Yo[4 * g + v][i_own] = y[v];
            if constexpr (KEEP) S.Uo[4 * g + v][i_own] = U[v];
        }
        const lds_t kb = kbs + (c & 1) * TWIN3;
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
            Sum2 x = SUM0;
            add32(x, get_twin(kb + TWIN_ROWS * jt), vu);
            St[jt] = St[jt] * ld4(dec + 16 * jt) + total(x);
        }
        __syncthreads();
    }
    store_rows(nch - 1);
    if (sT != nullptr) {
        float* dst = sT + static_cast<size_t>(i_own) * N + 4 * g;
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) st4(dst + 16 * jt, St[jt]);
    }
}

// KEEP: `s` and `sa` are written for a backward, 20 bytes per element beside the 14 of a bf16 forward's inputs and output.
// What bounds it: issue and, with KEEP, the writes (half of the states, and it takes 310 us instead of 332; fp32 mode 324 of 372).
// B8 T1024 C4096, one call, bf16: 398 us with every product on the fp32 matrix instructions, in four waves that did
// everything in turn between four barriers; 390 in two roles of four waves; 335 with split products but for the tiles, whose 16 fp32
// instructions a P wave held the vector unit for 512 cycles and took four more planes, twice the exponentials.  That form and the present one
// in alternation on one machine: bf16 329 -> 309 us, 273 -> 244 without KEEP; fp32 mode 377 -> 368, 310 -> 280 (2 to 4 us of that are
// exponentials and decays that are rounded once).
// Not kept: a ninth wave for the inverse (one workgroup a CU then: 502 us); rows asked for two chunks ahead (bf16 without KEEP 242 -> 253).
// Errors against 64 bits, T1024, fp32 mode, with the tiles on fp32 instructions -> now, 1e-7, at w = 0.5 +- 1, 2 +- 0.5, -3 +- 0.5, -6 +- 0.5, -8 +- 0.5:
// y 1.38 -> 0.80, 1.44 -> 0.78, 1.18 -> 0.96, 1.23 -> 1.16, 1.30 -> 1.22; sT 0.61 -> 0.55, 0.61 -> 0.56, 0.75 -> 0.69, 1.00 -> 0.96, 1.10 -> 1.04.
template <bool F32, bool KEEP, bool CUT>
__global__ __launch_bounds__(NTF, 4) void rwkv7c_fwd(const Args7c args) {
    const Args7c p = only_whole<CUT>(args);
    extern __shared__ __align__(32) unsigned char smem_raw[];
    SmemCF& S = *reinterpret_cast<SmemCF*>(smem_raw);
    const lds_t sb = lds_of(smem_raw);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const auto [bh, b, h] = head_of(p, blockIdx.x);
    Part7 x;
    if (!part_of(p, x)) return;
    const size_t tok0 = static_cast<size_t>(b) * p.T + x.first * CL;  // first token row of this block
    if (w < 4) {
        const int all = p.T / CL;
        const float* const s0 = x.n > 0 ? p.enter + (static_cast<size_t>(blockIdx.x) * (p.NB - 1) + x.n - 1) * N * N : first_state(p, p.s0, bh);
        float* const sT = p.sT != nullptr && x.first + x.chunks == all ? p.sT + bh * N * N : nullptr;
        fwd_role_s<F32, KEEP>(S, sb, p, s0, sT, KEEP ? p.s + (bh * all + x.first) * N * N : nullptr, w, tid, tok0, x.chunks, h);
    } else fwd_role_p<F32>(S, sb, p, w - 4, tid & 63, tok0, x.chunks, h);
}

// ---------------------------------------------------------------------------------------------------- blocks of time
// Few sequences: the heads' sequences in blocks, a workgroup each, in three launches.  A block takes the state S to S M + E, row by row:
// E is what it makes of an empty state, M of the identity without its own v; backwards the gradient state D becomes D M^T + F.  Both are
// one recurrence,  W = P1 S^T + T1 V, U = M0 W, S = S dec + U^T P2 + V^T P3,  per chunk:
//     forward   P1 = a e^{c_t}            T1 = AK     M0 = (I - AB)^{-1}  P2 = b e^{c_L - c_{s+1}}  P3 = k e^{c_L - c_{s+1}}  V = v
//     backward  P1 = b e^{c_L - c_{s+1}}  T1 = RB^T   M0 = (I - AB)^{-T}  P2 = a e^{c_t}            P3 = r e^{c_{t+1}}        V = dy
// (P1 S^T as in the kernels proper, P1 e^{-c_L} and S with the chunk's decay on it),
// which rwkv7c_local walks through (the roles of the forward without its outputs; a workgroup for E and one for M, which has no V).
// rwkv7c_scan takes the blocks in turn, 16 rows of a head a workgroup, on the fp32 matrix instructions.  M may overflow where the state
// itself is small (a, b that make it grow): a head with a scanned state that is not finite is walked through as a whole by the workgroup
// of its first block, as are heads with inputs that are no number.
struct SmemL {
    float AB[CL][TS];
    Decay part[4][N];
    float dec[2][N];
};
constexpr uint32_t L_S = (sizeof(SmemL) + 31) / 32 * 32, L_KB = L_S + PLANE3, L_V = L_KB + 2 * TWIN3;
template <bool F32> constexpr uint32_t L_MA = L_V + (F32 ? PLANE3 : TERM);
template <bool F32> constexpr uint32_t L_TOTAL = L_MA<F32> + TPAIR3;
static_assert(L_TOTAL<true> <= 80 * 1024, "two workgroups a CU");

template <bool F32, bool REV> DEVINL void local_role_p(SmemL& S, const lds_t sb, const Args7c& p, bool unit, int q, int lane, size_t tok0, int nch, int h) {
    const int l16 = lane & 15, g = lane >> 4, H = p.H;
    uint32_t nx[5][4];
    auto fetch = [&](int c) __attribute__((always_inline)) {
        c = c < nch ? c : nch - 1;
        const size_t base = ((tok0 + static_cast<size_t>(REV ? nch - 1 - c : c) * CL) * H + h) * N;
        uint32_t lo = lane;
        asm volatile("" : "+v"(lo));
        const uint16_t* const src[5] = {p.w, REV ? p.r : p.k, REV ? p.dy : p.v, p.a, p.b};
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int k = 0; k < 5; ++k) nx[k][e] = ld_raw<F32>(src[k], base, static_cast<uint32_t>((4 * q + e) * H) * N + lo);
    };
    Decay lam[4];
    float xx[4], aa[4], bb[4];
    uint32_t vb[4];
    auto convert = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            lam[e] = decay_of(widen<F32>(nx[0][e]));
            xx[e] = widen<F32>(nx[1][e]);
            vb[e] = unit ? 0u : nx[2][e];
            aa[e] = widen<F32>(nx[3][e]); bb[e] = widen<F32>(nx[4][e]);
        }
        S.part[q][lane] = sum4(lam);
    };
    auto planes = [&](const int slot) __attribute__((always_inline)) {
        float x[5], y[5];
        growth<!REV, REV && F32>(lam, S.part, q, lane, x, y);
        f32x4 p1, p2, p3;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p1[e] = REV ? bb[e] * y[e + 1] : aa[e] * y[e];
            p2[e] = REV ? aa[e] * x[e] : bb[e] * x[e + 1];
            p3[e] = xx[e] * x[e + 1];
        }
        const lds_t o = sb + piece(lane, q);
        put3(o + L_S, split3(p1));
        // (x is not above 1: what comes from bf16 inputs stays within bf16's range)
        put_twin(sb + L_KB + slot * TWIN3 + twin(lane, q), split3<!F32>(p3), split3<!F32>(p2));
        if constexpr (F32) put3(o + L_V, split3(f32x4{widen<F32>(vb[0]), widen<F32>(vb[1]), widen<F32>(vb[2]), widen<F32>(vb[3])}));
        else lds_st<u32x2>(o + L_V, u32x2{vb[0] | (vb[1] << 16), vb[2] | (vb[3] << 16)});
        if (q == 0) S.dec[slot][lane] = whole_decay(S.part, lane);
    };
    const Tr sp = tr_bases(sb + L_S, l16, g);
    const lds_t pp = tr_twin(sb + L_KB + (q == 0 ? 32 : 0), l16, g);
    fetch(0);
    convert();
    fetch(1);
    __syncthreads();
    planes(0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        if (q < 2) {
            auto one = [&](int hb) __attribute__((always_inline)) { return get3_tr(0, sp, hb); };
            auto pair = [&](int hb) __attribute__((always_inline)) { return get3_tr_twin(0, pp + (c & 1) * TWIN3, hb); };
            f32x4 x;
            if (q == 0) {
                f32x4 t;
                if constexpr (REV) t = causal_tile<false>(pair, one, true, l16, g) * UNHOLD;
                else t = causal_tile<false>(one, pair, true, l16, g) * UNHOLD;
                float m[CL];
                // (this wave wrote AB itself: LDS keeps a wave's accesses in order)
                if constexpr (REV) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) S.AB[4 * g + v][l16] = t[v];
                    inverse<false>(S.AB, l16, m);
                } else {
                    st4(&S.AB[l16][4 * g], t);
                    inverse<true>(S.AB, l16, m);
                }
                x = by_group(g, m);
            } else if constexpr (REV) x = causal_tile<false>(pair, one, false, l16, g);
            else x = causal_tile<true>(one, pair, true, l16, g);
            put_half<TTERM2>(sb + piece2(l16, g) + L_MA<F32> + (q == 0 ? 0 : 8), split3(x));
        }
        convert();
        fetch(c + 2);
        __syncthreads();
        planes((c + 1) & 1);
        __syncthreads();
    }
}
template <bool F32> DEVINL void local_role_s(SmemL& S, const lds_t sb, float* out, bool unit, int q, int lane, int nch) {
    const int l16 = lane & 15, g = lane >> 4, i_own = 16 * q + l16;
    f32x4 St[4];                                         // S[i_own][16 jt + 4 g + v]
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
#pragma unroll
        for (int v = 0; v < 4; ++v) St[jt][v] = unit && i_own == 16 * jt + 4 * g + v ? 1.f : 0.f;
    const Tr tr = tr_bases(sb, l16, g);
    const lds_t pp = sb + piece2(l16, g), vp = sb + L_V + piece(i_own, g), kbs = sb + L_KB + twin(l16, g);
    __syncthreads();
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const auto vop = [&]() __attribute__((always_inline)) { if constexpr (F32) return get3(vp); else return lds_ld<u32x2>(vp); }();
        const float* const dec = &S.dec[c & 1][4 * g];
        Sum2 W = SUM0;                                   // HOLD W
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
            add32(W, get3_tr(L_S, tr, hb), join(split3(St[2 * hb] * ld4(dec + 32 * hb)), split3(St[2 * hb + 1] * ld4(dec + 32 * hb + 16))));
        here(W);
        __syncthreads();
        add16(W, get_half<TTERM2>(pp + L_MA<F32> + 8), vop);
        Sum2 Us = SUM0;
        add16(Us, get_half<TTERM2>(pp + L_MA<F32>), split3(total(W) * UNHOLD));
        const Op3 vu = join(as3(vop), split3(total(Us)));
        const lds_t kb = kbs + (c & 1) * TWIN3;
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
            Sum2 x = SUM0;
            add32(x, get_twin(kb + TWIN_ROWS * jt), vu);
            St[jt] = St[jt] * ld4(dec + 16 * jt) + total(x);
        }
        __syncthreads();
    }
    float* const dst = out + static_cast<size_t>(i_own) * N + 4 * g;
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) st4(dst + 16 * jt, St[jt]);
}
template <bool F32, bool REV>
__global__ __launch_bounds__(NTF, 4) void rwkv7c_local(const Args7c p) {
    extern __shared__ __align__(32) unsigned char smem_raw[];
    SmemL& S = *reinterpret_cast<SmemL*>(smem_raw);
    const lds_t sb = lds_of(smem_raw);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = blockIdx.z >> 1, n = REV ? p.NB - 1 - m : m;
    const bool unit = blockIdx.z & 1;
    const auto [bh, b, h] = head_of(p, blockIdx.x);
    if (blockIdx.z == 0 && tid == 0) p.flags[blockIdx.x] = 0;
    const int chunks = min(p.per, p.T / CL - n * p.per);
    const size_t tok0 = static_cast<size_t>(b) * p.T + static_cast<size_t>(n) * p.per * CL;
    if (w < 4) local_role_s<F32>(S, sb, p.local + ((static_cast<size_t>(blockIdx.x) * (p.NB - 1) + m) * 2 + unit) * N * N, unit, w, tid & 63, chunks);
    else local_role_p<F32, REV>(S, sb, p, unit, w - 4, tid & 63, tok0, chunks, h);
}
// X_0 = s0 (backward: dsT), X_{m+1} = X_m M_m + E_m: a chain of NB - 1 small products; the next block's matrices are under way.
template <bool REV>
__global__ __launch_bounds__(256) void rwkv7c_scan(const Args7c p) {
    __shared__ float X[2][16][PS];
    const int tid = threadIdx.x, lane = tid & 63, q = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int rows = blockIdx.x & 3;
    const size_t head = blockIdx.x >> 2;
    const float* const init = REV ? p.dsT : p.s0;
    const uint32_t o = (16 * rows + 4 * g) * N + 16 * q + l16;       // element [4 g][16 q + l16] of these rows
    f32x4 x = ZERO4;
    if (init != nullptr)
#pragma unroll
        for (int v = 0; v < 4; ++v) x[v] = init[(p.at + head) * N * N + o + v * N];
    const float* at = p.local + head * (p.NB - 1) * 2 * N * N;
    float* to = p.enter + head * (p.NB - 1) * N * N + o;
    struct Block { float m[4][4]; f32x4 e; };
    auto fetch = [&](Block& d) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) d.m[s][e] = at[N * N + (16 * s + 4 * g + e) * N + 16 * q + l16];
#pragma unroll
        for (int v = 0; v < 4; ++v) d.e[v] = at[o + v * N];
    };
    Block now, next;
    fetch(now);
#pragma unroll
    for (int v = 0; v < 4; ++v) p.local[head * (p.NB - 1) * 2 * N * N + o + v * N] = x[v];      // (this thread has these elements of the first E; first_state)
    float bad = 0.f;
    for (int m = 0; m + 1 < p.NB; ++m, to += N * N) {
        if (m + 2 < p.NB) at += 2 * N * N;
        fetch(next);
#pragma unroll
        for (int v = 0; v < 4; ++v) X[m & 1][4 * g + v][16 * q + l16] = x[v];
        __syncthreads();
        f32x4 acc[2] = {now.e, ZERO4};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const f32x4 a = ld4(&X[m & 1][l16][16 * s + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[s & 1] = mm(a[e], now.m[s][e], acc[s & 1]);
        }
        x = acc[0] + acc[1];
#pragma unroll
        for (int v = 0; v < 4; ++v) { to[v * N] = x[v]; bad = fmaf(x[v], 0.f, bad); }
        now = next;
    }
    if (bad != 0.f) p.flags[head] = 1;                     // (0, or no number)
}

// ---------------------------------------------------------------------------------------------------- backward
// One workgroup of twelve waves per (batch, head), three roles with their own loops; wave w: q = w & 3.
//   waves 0..3 ("A", value-channel tile q): the gradient state, dS[jt][v] = dS[i = 16 q + l16][j = 16 jt + 4 g + v]   (rows j, columns i): the
//                B operand of the contractions over the key channel, B E^T and K E^T; dU, dW, dV, ds0, and the tiles dAB, dAK, dRB, dRK.
//   waves 4..7 ("B", key-channel tile q): the contractions over the value channel: U E and V E, with the split E of role A through LDS,
//                and dW S0, dY S0, with S0 of the chunk from `s`; they make dA, dR, dB, dK (register v <-> token 4 g + v, lane <-> key
//                channel), scale them, scan the decay gradient and park the results; they run one phase behind the A waves.
//   waves 8..11 ("P"): fetch the seven input rows and `sa` two chunks ahead, convert them, build the operand planes
//                (double-buffered), the causal tiles and the inverse.  The finished gradient rows leave LDS-staged, as whole rows, through the A waves.
// What bounds it: waits at the barriers, three a chunk, and issue.  Of 9400 cycles a chunk (B8 T1024 C4096, bf16 mode) a SIMD's vector unit has
// instructions for 5400 and its matrix unit for 2300, which overlap in part: neither is full, the roles wait for each other.  One call, bf16
// mode / fp32 mode, us: 762 / . with fp32 matrix instructions; 626 / 765 with split
// products but for the tiles, 11800 cycles a chunk, 5200 of them phase 3, where wave 0 of role A made a tile, an fp32 one and the inverse;
// 606 / 708 with inputs split once, the tiles with the P waves a phase earlier and what role B waited for with role A; 588 / 642 with one
// gradient state instead of two and the values that finish a chunk worked out in the phases before, in which role B waited; 564 / 634 now,
// with planes and an inverse that take fewer cycles; 4 us of that in either mode are exponentials and decays that are rounded once.
// Errors against 64 bits, T1024, fp32 mode, with the tiles on fp32 instructions -> now, 1e-7, at w = 0.5 +- 1, 2 +- 0.5, -3 +- 0.5, -6 +- 0.5, -8 +- 0.5:
// ds0 0.82 -> 0.76, 0.84 -> 0.80, 0.82 -> 0.75, 1.05 -> 1.02, 1.15 -> 1.09;
// dr 1.12 -> 0.90, 1.21 -> 0.88, 1.00 -> 0.97, 1.18 -> 1.14, 1.26 -> 1.20;
// dw 25.78 -> 20.69, 36.07 -> 25.50, 10.08 -> 9.55, 7.16 -> 6.86, 7.07 -> 6.65;
// dk 1.19 -> 0.93, 1.31 -> 0.91, 1.05 -> 1.03, 1.24 -> 1.22, 1.32 -> 1.27;
// dv 1.42 -> 0.93, 1.48 -> 0.91, 1.19 -> 1.02, 1.23 -> 1.22, 1.30 -> 1.27;
// da 1.88 -> 1.35, 2.03 -> 1.33, 1.62 -> 1.46, 1.76 -> 1.71, 1.90 -> 1.78;
// db 1.85 -> 1.30, 1.99 -> 1.28, 1.60 -> 1.47, 1.76 -> 1.71, 1.88 -> 1.79.
// (One w for all steps and channels, where a rounding repeats in every chunk: ds0 1.26 -> 1.14 at -4.3, 0.71 -> 0.72 at -1.)
constexpr int NTB = 12 * 64;       // waves 0..3 role A, 4..7 role B, 8..11 role P

constexpr int PK = 72;            // row stride (bf16 elements) of a parked output
// fp32 outputs are not parked (twice the bytes would not fit the CU's LDS): the waves that finish them store them from
// registers, 64 bytes of four rows per instruction.
template <bool F32>
struct SmemCB {
    Decay part[4][N];
    float dec[2][N];
    float AB[CL][TS];
    uint16_t park[F32 ? 1 : 5][F32 ? 1 : CL][F32 ? 1 : PK];                                // da, dr, db, dk, dw of the chunk that role B finished last, [token][channel]
    uint16_t parkv[F32 ? 1 : 2][F32 ? 1 : CL][F32 ? 1 : PK];                               // dv, which is ready one visit earlier than the other five
};
// A 64 x 64 matrix in bf16 terms, [i][j]: pieces of four j, turned by the row so that the writing lanes (16 rows by four pieces) and the
// transposing reads (8 rows of four pieces) meet every bank once.  i: of the first 16 rows, the others 2048 bytes on each
constexpr uint32_t DTERM = 64 * 128;
DEVINL lds_t square(int i, int piece) { return static_cast<lds_t>(128 * i + 8 * (piece ^ (4 * ((i >> 1) & 3)) ^ (2 * ((i >> 3) & 1)))); }
DEVINL bf16x8 tr16_square(lds_t o, int hb) {       // rows 32 hb + 16 (e >> 2) + 4 g + (e & 3) of a column
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef v4s __attribute__((address_space(3))) * ptr;
    const v4s x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(o + 4096 * hb)), y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(o + 4096 * hb + 2048));
    return op2(__builtin_bit_cast(u32x2, x), __builtin_bit_cast(u32x2, y));
}
// Planes and tiles behind it.  Two copies, of which the P waves fill one while the A and B waves work on the other: a e^{c_t} and
// r e^{c_{t+1}} (AR), b and k times HOLD e^{-c_{s+1}} (BK), U, v and dy (one term each where they are bf16) in three terms; fp32, 16 bytes of
// four tokens as the pairs lie: e^{c_{t+1}} (ES), W_SCALE sig (1 - sig) (DWF).  One: dS with the chunk's decay on it, in three terms (DS), dW, and the
// tiles, each as the lanes of its products hold it: the transposes of (I - AB)^{-1} and RB (MB), AK and RK (AKR); by rows (over s) dAB and
// dAK for dA, dRB and dRK for dR; by columns (over t) dAB and dRB for dB, dAK and dRK for dK.
template <bool F32> struct LB {
    static constexpr uint32_t TWO = (sizeof(SmemCB<F32>) + 31) / 32 * 32, EX = F32 ? PLANE3 : TERM;      // from TWO on
    static constexpr uint32_t AR = 0, BK = TWIN3, U = 2 * TWIN3, V = U + PLANE3, DY = V + EX, ES = DY + EX, DWF = ES + 4 * CL * N, SLOT = DWF + 4 * CL * N;
    static constexpr uint32_t ONE = (TWO + 2 * SLOT + 127) / 128 * 128;                                     // from ONE on
    static constexpr uint32_t DS = 0, DW = 3 * DTERM, MB = DW + PLANE3, AKR = MB + TPAIR3;
    static constexpr uint32_t A_ROWS = AKR + TPAIR3, R_ROWS = A_ROWS + TPAIR3, B_COLS = R_ROWS + TPAIR3, K_COLS = B_COLS + TPAIR3, BYTES = ONE + K_COLS + TPAIR3;
};
// A lane's addresses in one of the two regions
struct LaneB { Tr tr; lds_t own, pair, twin, own_twin; };
DEVINL LaneB lane_bases(lds_t base, int l16, int g, int own) {
    LaneB b{tr_bases(base, l16, g), base + piece(own, g), base + piece2(l16, g), base + rwkv::twin(l16, g), base + rwkv::twin(own, g)};
    opaque(b.tr.a); opaque(b.tr.b); opaque(b.own); opaque(b.pair); opaque(b.twin); opaque(b.own_twin);
    return b;
}
// The same lane's addresses in another region, d bytes on (modulo 2^32): an addition each, where bases of its own would be spilled
DEVINL LaneB moved(const LaneB& b, lds_t d) {
    return {{b.tr.a + d, b.tr.b + d}, b.own + d, b.pair + d, b.twin + d, b.own_twin + d};
}
// v, dy: four tokens of a channel, and over channels
template <bool F32> DEVINL auto exact_piece(lds_t a) { if constexpr (F32) return get3(a); else return lds_ld<u32x2>(a); }
template <bool F32> DEVINL auto exact_tr(uint32_t plane, const Tr& o, int hb) { if constexpr (F32) return get3_tr(plane, o, hb); else return ld_tr16(o, plane, hb); }
// causal_tile with planes chosen at run time, of three terms (or, not three, exact ones): rows of the result from a, columns from b; transposed: tokens s along
// the rows.  All but the planes' addresses is uniform: the waves that make different tiles share the code.
DEVINL f32x4 causal_split(const Tr& o, lds_t a, bool a3, lds_t b, bool b3, bool transposed, bool strict, int l16, int g) {
    Sum2 sum = SUM0;
    const Tr oa{o.a + a, o.b + a}, ob{o.a + b, o.b + b};
    const bf16x8 ah[2] = {ld_tr16(oa, 0, 0), ld_tr16(oa, 0, 1)}, bh[2] = {ld_tr16(ob, 0, 0), ld_tr16(ob, 0, 1)};
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) sum.hi = mmb(ah[hb], bh[hb], sum.hi);
    if (a3) {
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const bf16x8 am = ld_tr16(oa, TERM, hb);
            sum.lo = mmb(ld_tr16(oa, 2 * TERM, hb), bh[hb], sum.lo);
            if (b3) sum.lo = mmb(am, ld_tr16(ob, TERM, hb), sum.lo);
            sum.lo = mmb(am, bh[hb], sum.lo);
        }
    }
    if (b3) {
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) sum.lo = mmb(ah[hb], ld_tr16(ob, TERM, hb), mmb(ah[hb], ld_tr16(ob, 2 * TERM, hb), sum.lo));
    }
    f32x4 acc = total(sum);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 4 * g + v, t = transposed ? l16 : r, s = transposed ? r : l16;
        acc[v] = (strict ? s < t : s <= t) ? acc[v] : 0.f;
    }
    return acc;
}

// Per visit i (chunks in descending order) every wave passes three barriers; role B finishes a visit in the next one's phase 1, so that all
// roles always have matrix work in the same phase.  What they do, and what of LDS they read (<) and write (>) between two barriers; (i): the
// copy of visit i of what has two:
//     phase 1   A   B E^T, K E^T of i                                                < BK (i), dec (i)                       > DS
//               B   dA, dB, dK and what is left of i - 1                             < A_ROWS, B_COLS, K_COLS, DWF (i - 1)   > park
//               P   planes of i + 1                                                  < part                                  > AR, BK, U, V, DY, dec (i + 1)
//     phase 2   A   dU, dW, dV, the state of i; the tiles dRB, dRK of i to LDS       < MB, AKR, AR, DY, V (i), dec (i)       > DW, R_ROWS, B_COLS and K_COLS (dRB, dRK), parkv (i)
//               B   dY S0, U E, V E of i; AR, BK of i into registers                 < DS, AR, BK, U, V, DY (i)
//               P   the causal tiles of i + 1; factors; decays of i + 2              < AR, BK (i + 1)                        > ES, DWF (i + 1), part
//     phase 3   A   dAB, dAK of i, dRB, dRK of i + 1; rows of i - 1 to memory        < DW, U, V (i), DY, U, V (i + 1), park, parkv (i - 1)   > A_ROWS, B_COLS and K_COLS (dAB, dAK)
//               B   dW S0, dR of i; the state entering the next chunk asked for      < DW, R_ROWS, ES (i)
//               P   the inverse and the tiles of i + 1 to LDS; rows of i + 4 asked for                                       > AB, MB, AKR
// (In visit 0 role B has P at the end of the call to make in phase 1, from U, V, BK and dec of visit 0.)

// ---- role P: elementwise preparation (lane = channel, tokens 4 wp + e) one visit ahead, and the row-wise output stores
struct Prep7 { uint32_t nx[7][4]; float nsa[4]; };
template <bool F32> struct Conv7 { float sg[4], uu[4]; Decay lam[4]; uint32_t pk[6][F32 ? 4 : 2]; };   // sigmoid(w), sa, and r k v a b dy: fp32, or bf16 pairs (tokens 2 z, 2 z + 1)
template <bool F32> DEVINL void bwd_fetch(const Args7c& p, Prep7& x, size_t row0, int wp, int lane, int H, int h) {
    // wave-uniform base (scalar registers) plus a 32-bit lane offset: no 64-bit address per tensor and token in vector registers
    // (the lane part is hidden from the optimiser: it would otherwise turn every tensor-and-token address into a 64-bit
    // induction variable of the chunk loop, 64 vector registers)
    const size_t base = (row0 * H + h) * N;
    uint32_t lo = lane;
    asm volatile("" : "+v"(lo));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t o = static_cast<uint32_t>((4 * wp + e) * H) * N + lo;
        const uint16_t* const src[7] = {p.w, p.r, p.k, p.v, p.a, p.b, p.dy};
#pragma unroll
        for (int k = 0; k < 7; ++k) x.nx[k][e] = ld_raw<F32>(src[k], base, o);
        x.nsa[e] = (p.sa + base)[o];
    }
}
// first half of the preparation: the decay of each token, this wave's decay sum; the other inputs are kept packed so that the
// registers of x are free for the next fetch
template <bool F32> DEVINL void bwd_convert(Decay (*part)[N], const Prep7& x, Conv7<F32>& y, int wp, int lane) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        y.sg[e] = sigmoid_fast(widen<F32>(x.nx[0][e]));
        y.lam[e] = decay_of_sig(y.sg[e]);
        y.uu[e] = x.nsa[e];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        if constexpr (F32) {
#pragma unroll
            for (int e = 0; e < 4; ++e) y.pk[k][e] = x.nx[k + 1][e];
        } else {
#pragma unroll
            for (int z = 0; z < 2; ++z) y.pk[k][z] = x.nx[k + 1][2 * z] | (x.nx[k + 1][2 * z + 1] << 16);
        }
    }
    part[wp][lane] = sum4(y.lam);
}
// second half (after a barrier), in two parts: what the factors enter; the rest
template <bool F32> struct In7 {
    const Conv7<F32>& y;
    DEVINL float operator()(int k, int e) const {
        if constexpr (F32) return __uint_as_float(y.pk[k][e]);
        else return (e & 1) ? bf_hi(y.pk[k][e >> 1]) : bf_lo(y.pk[k][e >> 1]);
    }
};
// sb: LDS base, slot: offset of the chunk's copy, dec: of the chunk
template <bool F32> DEVINL f32x4 bwd_planes(const lds_t sb, const lds_t slot, float* dec, const Decay (*part)[N], const Conv7<F32>& y, int wp, int lane) {
    using O = LB<F32>;
    float x[5], i[5];
    growth<false, F32>(y.lam, part, wp, lane, x, i);
    const In7<F32> in{y};
    f32x4 as, rs, bs, ks;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        as[e] = in(3, e) * x[e];
        rs[e] = in(0, e) * x[e + 1];
        bs[e] = in(4, e) * i[e + 1];
        ks[e] = in(1, e) * i[e + 1];
    }
    // (rounded products: a remainder fused with one would put into the planes what role B's factors do not hold)
    asm volatile("" : "+v"(as), "+v"(rs), "+v"(bs), "+v"(ks));
    const lds_t o = sb + O::TWO + slot + twin(lane, wp);
    // (x is not above 1: what comes from bf16 inputs stays within bf16's range)
    put_twin(o + O::AR, split3<!F32>(as), split3<!F32>(rs));
    put_twin(o + O::BK, split3(bs), split3(ks));
    if (wp == 0) dec[lane] = whole_decay(part, lane);
    return {x[1], x[2], x[3], x[4]};
}
template <bool F32> DEVINL void bwd_planes_rest(const lds_t sb, const lds_t slot, const f32x4& es, const Conv7<F32>& y, int wp, int lane) {
    using O = LB<F32>;
    const lds_t o = sb + O::TWO + slot;
    lds_st<f32x4>(o + O::ES + piece2(lane, wp), es);
    f32x4 f;
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = W_SCALE * y.sg[e] * (1.f - y.sg[e]);
    lds_st<f32x4>(o + O::DWF + piece2(lane, wp), f);
}
// U, v and dy, which no factor enters
template <bool F32> DEVINL void bwd_planes_raw(const lds_t sb, const lds_t slot, const Conv7<F32>& y, int wp, int lane) {
    using O = LB<F32>;
    const In7<F32> in{y};
    const lds_t o = sb + O::TWO + slot + piece(lane, wp);
    put3(o + O::U, split3(f32x4{y.uu[0], y.uu[1], y.uu[2], y.uu[3]}));
    if constexpr (F32) {
        put3(o + O::V, split3(f32x4{in(2, 0), in(2, 1), in(2, 2), in(2, 3)}));
        put3(o + O::DY, split3(f32x4{in(5, 0), in(5, 1), in(5, 2), in(5, 3)}));
    } else {
        lds_st<u32x2>(o + O::V, u32x2{y.pk[2][0], y.pk[2][1]});
        lds_st<u32x2>(o + O::DY, u32x2{y.pk[5][0], y.pk[5][1]});
    }
}
// bf16: da dr db dk dw (and dv) of one chunk leave their parking places as whole rows (256 threads, four channels each)
DEVINL void bwd_store_rows(const SmemCB<false>& S, int vbuf, const Args7c& p, size_t row0, int tp, int H, int h) {
    const int t = tp >> 4, c4 = (tp & 15) * 4;
    const size_t base = (row0 * H + h) * N;
    uint32_t o = static_cast<uint32_t>(t * H) * N + c4;
    asm volatile("" : "+v"(o));
    auto put = [&](uint16_t* dst, const uint16_t* src) __attribute__((always_inline)) {
        *reinterpret_cast<uint2*>(dst + base + o) = *reinterpret_cast<const uint2*>(src);
    };
    put(p.da, &S.park[0][t][c4]); put(p.dr, &S.park[1][t][c4]); put(p.db, &S.park[2][t][c4]); put(p.dk, &S.park[3][t][c4]);
    put(p.dw, &S.park[4][t][c4]); put(p.dv, &S.parkv[vbuf][t][c4]);
}
// fp32: element `first` + o straight to global memory.  (One scalar base a tensor and the row in the lane's offset: with a base for each
// of the twenty rows that a B wave stores the scalar registers were spilled.)
DEVINL void store_f32(uint16_t* dst, size_t first, uint32_t o, float x) {
    *reinterpret_cast<float*>(reinterpret_cast<char*>(dst) + first * 4 + o * 4u) = x;
}
template <bool F32> DEVINL void bwd_role_p(SmemCB<F32>& S, const lds_t sb, const Args7c& p, int tid, int w, size_t tok0, int nch, int H, int h) {
    const int lane = tid & 63, wp = w - 8;
    // Raw rows are asked for two visits before they are converted (one visit, of which only two phases lie between the
    // request and the use, is less than the memory system takes under load: the A and B waves then waited for the P waves
    // at two of the three barriers of every visit).  Two register sets take turns; the chunk index is clamped instead of
    // the request being skipped, so that every visit issues the same loads and the waits count the same.
    Prep7 x[2];
    Conv7<F32> y;
    const int l16 = lane & 15, g = lane >> 4;
    using L = LB<F32>;
    const lds_t tp = tr_twin(sb, l16, g);
    // a causal tile of a visit
    auto tile = [&](const int visit) __attribute__((always_inline)) {
        const lds_t at = tp + L::TWO + (visit & 1) * L::SLOT;
        return causal_tile<false>([&](int hb) __attribute__((always_inline)) { return get3_tr_twin(0, at + (wp < 2 ? L::AR : L::AR + 32), hb); },
                                  [&](int hb) __attribute__((always_inline)) { return get3_tr_twin(0, at + (wp & 1 ? L::BK + 32 : L::BK), hb); }, wp < 2, l16, g);
    };
    // its place, of AB the inverse's
    auto put_tile = [&](const f32x4& acc) __attribute__((always_inline)) {
        f32x4 x = acc;
        if (wp == 0) {                           // this wave wrote AB itself: LDS keeps a wave's accesses in order
#pragma unroll
            for (int v = 0; v < 4; ++v) S.AB[4 * g + v][l16] = acc[v] * UNHOLD;
            float m[CL];
            inverse<false>(S.AB, l16, m);
                x = by_group(g, m);
        }
        // (one store with a selected address: with one in each of the branches the compiler merged them and left the address undefined
        // on one way there)
        put_half<TTERM2>(sb + L::ONE + piece2(l16, g) + (wp == 0 ? L::MB : (wp == 1 ? L::AKR : (wp == 2 ? L::MB + 8 : L::AKR + 8))), split3(x));
    };
    auto row_of = [&](int visit) { const int c = nch - 1 - visit; return tok0 + static_cast<size_t>(c > 0 ? c : 0) * CL; };
    bwd_fetch<F32>(p, x[0], row_of(0), wp, lane, H, h);
    bwd_fetch<F32>(p, x[1], row_of(1), wp, lane, H, h);
    bwd_convert(S.part, x[0], y, wp, lane);           // visit 0, before the loop
    bwd_fetch<F32>(p, x[0], row_of(2), wp, lane, H, h);
    __syncthreads();
    bwd_planes_rest<F32>(sb, 0, bwd_planes<F32>(sb, 0, S.dec[0], S.part, y, wp, lane), y, wp, lane);
    bwd_planes_raw<F32>(sb, 0, y, wp, lane);
    __syncthreads();
    put_tile(tile(0));
    if (nch > 1) bwd_convert(S.part, x[1], y, wp, lane);
    bwd_fetch<F32>(p, x[1], row_of(3), wp, lane, H, h);
    __syncthreads();
    auto visit = [&](const int i, auto Z) __attribute__((always_inline)) {     // visit i is chunk nch - 1 - i
        constexpr int z = decltype(Z)::value;        // the set that holds visit i + 2
        const bool next = i + 1 < nch;
        const lds_t slot = ((i + 1) & 1) * L::SLOT;
        f32x4 es = ZERO4, t = ZERO4;
        if (next) {
            es = bwd_planes<F32>(sb, slot, S.dec[(i + 1) & 1], S.part, y, wp, lane);
            bwd_planes_raw<F32>(sb, slot, y, wp, lane);
        }
        __syncthreads();
        if (next) {
            t = tile(i + 1);
            bwd_planes_rest<F32>(sb, slot, es, y, wp, lane);
        }
        if (i + 2 < nch) bwd_convert(S.part, x[z], y, wp, lane);
        __syncthreads();
        if (next) put_tile(t);
        bwd_fetch<F32>(p, x[z], row_of(i + 4), wp, lane, H, h);
        __syncthreads();
    };
    for (int i = 0; i < nch; i += 2) {
        visit(i, std::integral_constant<int, 0>{});
        if (i + 1 < nch) visit(i + 1, std::integral_constant<int, 1>{});
    }
    __syncthreads();                                 // role B finishes the last chunk
    if constexpr (!F32) bwd_store_rows(S, (nch - 1) & 1, p, tok0, tid - 8 * 64, H, h);
}

template <bool F32> DEVINL void bwd_role_a(SmemCB<F32>& S, const lds_t sb, const Args7c& p, const float* dsT, float* ds0, int tid, int w, int nch, size_t tok0, int H, int h) {
    const int lane = tid & 63, q = w & 3, l16 = lane & 15, g = lane >> 4;
    const int own = 16 * q + l16;                    // value channel i of this lane's column
    f32x4 dS[4];                                     // dS[i = own][j = 16 jt + 4 g + v]
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
        dS[jt] = dsT != nullptr ? ld4(dsT + static_cast<size_t>(own) * N + 16 * jt + 4 * g) : ZERO4;
    using L = LB<F32>;
    const LaneB one = lane_bases(sb + L::ONE, l16, g, own);
    const Tr base_tr = tr_bases(sb, l16, g);
    const lds_t tp = tr_twin(sb, l16, g);
    const lds_t sq = sb + L::ONE + L::DS + square(own, g);
    auto put_square = [&](int jt, const B3& x) __attribute__((always_inline)) {
        const lds_t o = sq ^ (32u * jt);             // (128-byte rows, and the piece's upper bits are turned by exclusive or)
        lds_st<u32x2>(o, x.h); lds_st<u32x2>(o + DTERM, x.m); lds_st<u32x2>(o + 2 * DTERM, x.l);
    };
    // dRB (q odd), dRK, by rows and by columns, of a visit, made in the one before.  (With U, the longer ones where v is one term, on the odd
    // waves: the inverse runs beside wave 0.)
    const bool byrow = q < 2, uv3 = F32 || (q & 1) != 0;
    auto uv_of = [&](int visit) __attribute__((always_inline)) { return L::TWO + (visit & 1) * L::SLOT + (q & 1 ? L::U : L::V); };
    auto dr_tile = [&](int visit) __attribute__((always_inline)) {
        const lds_t y = L::TWO + (visit & 1) * L::SLOT + L::DY, uv = uv_of(visit);
        f32x4 t = causal_split(base_tr, byrow ? uv : y, byrow ? uv3 : F32, byrow ? y : uv, byrow ? F32 : uv3, byrow, false, l16, g);
        asm volatile("" : "+v"(t));
        return t;
    };
    __syncthreads();
    __syncthreads();
    f32x4 dr = dr_tile(0);
    __syncthreads();
    for (int i = 0; i < nch; ++i) {
        const LaneB two = moved(one, L::TWO + (i & 1) * L::SLOT - L::ONE);
        const float* const dec = &S.dec[i & 1][4 * g];
        // ---------------------------------------------------------------- phase 1: the parts of dU, dV that need no tile
        Sum2 dUs = SUM0, dVs = SUM0;                     // HOLD dU, HOLD dV
        const lds_t bk = tp + L::TWO + (i & 1) * L::SLOT + L::BK;
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            // (decayed for these products only: in the update a fused multiplication and addition rounds the state once)
            const B3 s0 = split3(dS[2 * hb] * ld4(dec + 32 * hb)), s1 = split3(dS[2 * hb + 1] * ld4(dec + 32 * hb + 16));
            put_square(2 * hb, s0); put_square(2 * hb + 1, s1);      // for role B
            const Op3 st = join(s0, s1);
            add32(dUs, get3_tr_twin(0, bk, hb), st);
            add32(dVs, get3_tr_twin(32, bk, hb), st);
        }
        here(dUs); here(dVs);
        __syncthreads();
        // ---------------------------------------------------------------- phase 2: dU, dW = M^T dU, dV, the gradient state
        {
            const auto dyop = exact_piece<F32>(two.own + L::DY);             // dY[tau = 4 g + v][i]
            add16(dUs, get_half<TTERM2>(one.pair + L::MB + 8), dyop);
            Sum2 dWs = SUM0;
            add16(dWs, get_half<TTERM2>(one.pair + L::MB), split3(total(dUs) * UNHOLD));
            const B3 dW = split3(total(dWs));
            put3(one.own + L::DW, dW);
            const Op3 wy = join(dW, as3(dyop));          // dW and dY share the instructions of what follows
            add32(dVs, get_pair<TTERM2>(one.pair + L::AKR), wy);
            const f32x4 dV = total(dVs) * UNHOLD;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (F32) store_f32(p.dv, ((tok0 + static_cast<size_t>(nch - 1 - i) * CL) * H + h) * N, static_cast<uint32_t>((4 * g + v) * H) * N + own, dV[v]);
                else S.parkv[i & 1][4 * g + v][own] = f2bf(dV[v]);
            }
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) {
                Sum2 x = SUM0;
                add32(x, get_twin(two.twin + L::AR + TWIN_ROWS * jt), wy);
                dS[jt] = dS[jt] * ld4(dec + 16 * jt) + total(x);
            }
            put_half<TTERM2>(one.pair + (q == 1 ? L::R_ROWS : (q == 0 ? L::R_ROWS + 8 : (q == 3 ? L::B_COLS + 8 : L::K_COLS + 8))), split3(dr));
        }
        __syncthreads();
        // ---------------------------------------------------------------- phase 3: dAB (q odd), dAK (they need dW), by rows and by columns
        {
            const lds_t w = L::ONE + L::DW, uv = uv_of(i);
            const f32x4 t = causal_split(base_tr, byrow ? uv : w, byrow ? uv3 : true, byrow ? w : uv, byrow ? true : uv3, byrow, true, l16, g);
            put_half<TTERM2>(one.pair + (q == 1 ? L::A_ROWS : (q == 0 ? L::A_ROWS + 8 : (q == 3 ? L::B_COLS : L::K_COLS))), split3(t));
        }
        if (i + 1 < nch) dr = dr_tile(i + 1);
        // These waves carry the finished rows of the visit before to global memory (parked by the B waves in phase 1, dv by this role one
        // visit earlier; both stay as they are until the next visit).
        if constexpr (!F32) {
            if (i > 0) bwd_store_rows(S, (i - 1) & 1, p, tok0 + static_cast<size_t>(nch - i) * CL, tid, H, h);
        }
        __syncthreads();
    }
    __syncthreads();
    if (ds0 != nullptr) {
        float* dst = ds0 + static_cast<size_t>(own) * N + 4 * g;
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) st4(dst + 16 * jt, dS[jt]);
    }
}

// The lane's number, worked out where it is used.  (What is derived from threadIdx is kept in registers across the chunk loop, and where
// those do not last, in scratch: a reload waits for all loads under way, the next state among them.)
DEVINL uint32_t lane_again() {
    uint32_t all = ~0u;
    asm volatile("" : "+s"(all));
    return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u));
}
template <bool F32> DEVINL void bwd_role_b(SmemCB<F32>& S, const lds_t sb, const Args7c& p, const float* dsT, const float* slots, int tid, int w, int nch, size_t tok0, int H, int h) {
    const int lane = tid & 63, q = w & 3, l16 = lane & 15, g = lane >> 4;
    const int own = 16 * q + l16;                    // key channel j of this lane's column
    using L = LB<F32>;
    LaneB one = lane_bases(sb + L::ONE, l16, g, own);
    f32x4 S0b[4];                                    // S0 at [i = 16 ib + 4 g + v][j = own]
    auto fetch_state = [&](int c) __attribute__((always_inline)) {
        const float* slot = slots + static_cast<size_t>(c) * N * N;
        const uint32_t me = lane_again();
        const uint32_t o = ((me >> 4) * (4 * N) + 16 * q + (me & 15)) * 4u;
        const char* const at = reinterpret_cast<const char*>(slot);
#pragma unroll
        for (int ib = 0; ib < 4; ++ib)
#pragma unroll
            for (int v = 0; v < 4; ++v) S0b[ib][v] = *reinterpret_cast<const float*>(at + (16 * ib + v) * N * 4 + o);
    };
    [[maybe_unused]] lds_t park = sb + static_cast<uint32_t>(offsetof(SmemCB<F32>, park)) + static_cast<uint32_t>(4 * g * PK + own) * 2;      // parked outputs
    opaque(park);
    // (addresses worked out where they are used: kept in registers, others go to scratch)
    auto decay_of = [&](int visit) __attribute__((always_inline)) {
        return lds_ld<float>(sb + static_cast<uint32_t>(offsetof(SmemCB<F32>, dec)) + 64 * q + (visit & 1) * 4 * N + 4 * (lane_again() & 15));
    };
    // piece of channel l16; of channel 16 ib + l16, 512 ib on, it is turned by two groups where ib is odd
    auto rows = [&]() __attribute__((always_inline)) { const uint32_t me = lane_again(); return piece(me & 15, me >> 4); };
    auto copy_of = [&](int visit) __attribute__((always_inline)) { return static_cast<lds_t>(L::TWO + (visit & 1) * L::SLOT); };
    float Pj = 0.f;                                  // P at the end of the chunk that is finished next
    f32x4 xA = ZERO4, xB = ZERO4, xK = ZERO4, dRp = ZERO4;    // state parts of dA, dB, dK, and dR, carried into the next visit's phase 1
    // and of the planes of the own channel, whose places the P waves fill anew there, operands and values; e^{c_{t+1}}, before the first
    // of the four tokens e^{c_t}, HOLD e^{-c_{t+1}}
    Op3 ar, bk;
    f32x4 va, vr, vb, vk, er, eb;
    float ea0 = 1.f;
    // a contraction over 16 with a pair of tiles (one after the other: the registers do not hold the operands of all of them)
    auto tile2 = [&](uint32_t pair, const Op3& b) __attribute__((always_inline)) {
        Sum2 s = SUM0;
        add32(s, get_pair<TTERM2>(one.pair + pair), b);
        __builtin_amdgcn_sched_barrier(0);
        return total(s);
    };
    // the values that a side of an operand holds.  (Those, and not inputs times factors, go into the sums for the decay gradient: what of
    // one product is in another cancels there.)
    auto value = [&](const Op3& o, const int side) __attribute__((always_inline)) {
        f32x4 x;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t h = __builtin_bit_cast(u32x4, o.h)[2 * side + w], m = __builtin_bit_cast(u32x4, o.m)[2 * side + w], l = __builtin_bit_cast(u32x4, o.l)[2 * side + w];
            x[2 * w] = bf_lo(h) + (bf_lo(m) + bf_lo(l));
            x[2 * w + 1] = bf_hi(h) + (bf_hi(m) + bf_hi(l));
        }
        return x;
    };
    // tile parts, scaling, decay gradient of the chunk of a visit, whose first row is row0; results parked as bf16
    auto finish = [&](const int visit, const size_t row0) __attribute__((always_inline)) {
        const uint32_t me = lane_again();
        [[maybe_unused]] const uint32_t lo = (me >> 4) * static_cast<uint32_t>(4 * H * N) + 16 * q + (me & 15);
        [[maybe_unused]] const size_t first = (row0 * H + h) * N;
        auto put = [&](const int k, uint16_t* dst, const int v, const float x) __attribute__((always_inline)) {
            if constexpr (F32) store_f32(dst, first, lo + static_cast<uint32_t>(v * H) * N, x);
            else lds_st<uint16_t>(park + 2 * PK * (CL * k + v), f2bf(x));
        };
        const f32x4 tA = tile2(L::A_ROWS, bk);
        const f32x4 tB = tile2(L::B_COLS, ar), tK = tile2(L::K_COLS, ar);
        const f32x4 dwf = lds_ld<f32x4>(sb + copy_of(visit) + L::DWF + piece2(16 * q + (me & 15), me >> 4));
        float del[4], ada[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float dAp = fmaf(UNHOLD, tA[v], xA[v]), dBp = tB[v] + xB[v], dKp = tK[v] + xK[v];
            put(0, p.da, v, dAp * (v == 0 ? ea0 : er[v - 1]));
            put(1, p.dr, v, dRp[v] * er[v]);
            put(2, p.db, v, dBp * (eb[v] * UNHOLD));
            put(3, p.dk, v, dKp * (eb[v] * UNHOLD));
            ada[v] = va[v] * dAp;
            del[v] = fmaf(vr[v], dRp[v], -UNHOLD * fmaf(vk[v], dKp, vb[v] * dBp));      // r dr - b db - k dk
        }
        // G_t = P_{t+1} + del_t,  P_t = G_t + a da:  suffix sums over t = 4 g + v, later lane groups first
        const float tot = ((del[0] + ada[0]) + (del[1] + ada[1])) + ((del[2] + ada[2]) + (del[3] + ada[3]));
        auto of_lane = [](uint32_t l, float x) __attribute__((always_inline)) { return __int_as_float(__builtin_amdgcn_ds_bpermute(static_cast<int>(4 * l), __float_as_int(x))); };
        const float t1 = of_lane(me + 16, tot), t2 = of_lane(me + 32, tot), t3 = of_lane(me + 48, tot);
        float Pn = Pj + ((me < 48 ? t1 : 0.f) + ((me < 32 ? t2 : 0.f) + (me < 16 ? t3 : 0.f)));     // P after this lane's last token
#pragma unroll
        for (int v = 3; v >= 0; --v) {
            const float G = Pn + del[v];
            Pn = G + ada[v];
            put(4, p.dw, v, G * dwf[v]);
        }
        Pj = of_lane(me & 15, Pn);                   // lane group 0 holds P at the start of the chunk
    };
    fetch_state(nch - 1);
    __syncthreads();
    __syncthreads();
    __syncthreads();
    for (int i = 0; i < nch; ++i) {
        const int c = nch - 1 - i;
        const LaneB two = moved(one, copy_of(i) - L::ONE);
        // ---------------------------------------------------------------- phase 1: finish the previous visit's chunk
        if (i > 0) finish(i - 1, tok0 + static_cast<size_t>(c + 1) * CL);
        else if (dsT != nullptr) {
            // P at the end of the call: sum_i dsT o S_T with S_T = (S0 + U^T (b e^{-c_{s+1}}) + V^T (k e^{-c_{s+1}})) dec of the last chunk
            const float decj = decay_of(i);
            const Op3 bk = get_twin(two.own_twin + L::BK);
            const lds_t row = rows();
            float pp = 0.f;
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) {
                const lds_t o = sb + copy_of(i) + (row ^ (ib & 1 ? 16u : 0u)) + 512 * ib;
                Sum2 x = SUM0;
                add32(x, join(get3(o + L::U), as3(exact_piece<F32>(o + L::V))), bk);
                const f32x4 acc = total(x);
#pragma unroll
                for (int v = 0; v < 4; ++v) pp = fmaf(dsT[(16 * ib + 4 * g + v) * N + own], fmaf(acc[v], UNHOLD, S0b[ib][v]) * decj, pp);
            }
            pp += __shfl_xor(pp, 16, 64);
            pp += __shfl_xor(pp, 32, 64);
            Pj = pp;
        }
        __syncthreads();
        // ---------------------------------------------------------------- phase 2: dY S0, U E, V E
        auto dy_of = [&](int hb) __attribute__((always_inline)) { return exact_tr<F32>(L::DY, two.tr, hb); };
        auto u_of = [&](int hb) __attribute__((always_inline)) { return get3_tr(L::U, two.tr, hb); };
        auto v_of = [&](int hb) __attribute__((always_inline)) { return exact_tr<F32>(L::V, two.tr, hb); };
        Op3 s0[2];
        f32x4 xR;
        ar = get_twin(two.own_twin + L::AR); bk = get_twin(two.own_twin + L::BK);
        va = value(ar, 0); vr = value(ar, 1); vb = value(bk, 0); vk = value(bk, 1);
        asm volatile("" : "+v"(va), "+v"(vr), "+v"(vb), "+v"(vk));            // (here, or the compiler takes all this to where it is used)
        {
            Sum2 pr = SUM0, pb = SUM0, pk = SUM0;
            const lds_t sq = sb + L::ONE + L::DS + square(4 * g + (l16 >> 2), 4 * q + (l16 & 3));
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
                s0[hb] = join(split3(S0b[2 * hb]), split3(S0b[2 * hb + 1]));
                const Op3 ds = {tr16_square(sq, hb), tr16_square(sq + DTERM, hb), tr16_square(sq + 2 * DTERM, hb)};      // dS dec, of role A
                add32(pr, dy_of(hb), s0[hb]);
                add32(pb, u_of(hb), ds);
                add32(pk, v_of(hb), ds);
            }
            xR = total(pr); xB = total(pb); xK = total(pk);
        }
        __syncthreads();
        // ---------------------------------------------------------------- phase 3: dW S0, dR
        {
            const uint32_t me = lane_again();
            er = lds_ld<f32x4>(sb + copy_of(i) + L::ES + piece2(16 * q + (me & 15), me >> 4));
            ea0 = lds_ld<float>(sb + copy_of(i) + L::ES + 12 + piece2(16 * q + (me & 15), me > 15 ? (me >> 4) - 1 : 0));
            if (me < 16) ea0 = 1.f;
#pragma unroll
            for (int v = 0; v < 4; ++v) eb[v] = held_inverse<F32>(er[v]);                    // (er is between e^-9.8 and 1)
            asm volatile("" : "+v"(er), "+v"(eb), "+v"(ea0));
            Sum2 pa = SUM0;
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) add32(pa, get3_tr(L::DW, one.tr, hb), s0[hb]);
            xA = total(pa);
            // dR needs no tile of this phase
            const f32x4 tR = tile2(L::R_ROWS, bk);
#pragma unroll
            for (int v = 0; v < 4; ++v) dRp[v] = fmaf(UNHOLD, tR[v], xR[v]);
            if (c > 0) fetch_state(c - 1);
        }
        __syncthreads();
    }
    opaque(one.pair);                                // (or the tiles' addresses are kept from before the loop, in scratch)
    finish(nch - 1, tok0);
    __syncthreads();
}

template <bool F32, bool CUT>
__global__ __launch_bounds__(NTB, 3) void rwkv7c_bwd(const Args7c args) {
    const Args7c p = only_whole<CUT>(args);
    extern __shared__ __align__(128) unsigned char smem_raw[];
    SmemCB<F32>& S = *reinterpret_cast<SmemCB<F32>*>(smem_raw);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const auto [bh, b, h] = head_of(p, blockIdx.x);
    Part7 x;
    if (!part_of(p, x)) return;
    const size_t tok0 = static_cast<size_t>(b) * p.T + x.first * CL;
    const int nch = x.chunks, all = p.T / CL;
    const lds_t sb = lds_of(smem_raw);
    // (thread numbers anew: role B has no register to hold one across its loop for the code of the others, which lies behind)
    const auto again = [&]() __attribute__((always_inline)) { return 64 * w + static_cast<int>(lane_again()); };
    if (w >= 8) { bwd_role_p(S, sb, p, again(), w, tok0, nch, p.H, h); return; }
    const float* const dsT = x.first + nch < all ? p.enter + (static_cast<size_t>(blockIdx.x) * (p.NB - 1) + p.NB - 2 - x.n) * N * N : first_state(p, p.dsT, bh);
    if (w < 4) bwd_role_a(S, sb, p, dsT, p.ds0 != nullptr && x.n == 0 ? p.ds0 + bh * N * N : nullptr, again(), w, nch, tok0, p.H, h);
    else bwd_role_b(S, sb, p, dsT, p.s + (bh * all + x.first) * N * N, tid, w, nch, tok0, p.H, h);
}

const uint16_t* el(const void* p) { return static_cast<const uint16_t*>(p); }
uint16_t* el(void* p) { return static_cast<uint16_t*>(p); }

// Blocks of time: as many as there is room for on the card at a time (two workgroups a CU in the forward, one in the backward), of
// BLOCK_CHUNKS chunks at least; 1: whole sequences.  per: chunks a block.  The first pass does the work of a forward without its outputs
// twice, which pays where a whole sequence leaves most of the card idle.  Where the line lies, heads, us whole / in blocks, bf16
// forward: 8 of T256 41 / 30, of T4096 588 / 104; 64 of T256 41 / 40, of T4096 598 / 345; 128 of T1024 153 / 163, of T4096 626 / 591; 192 in two blocks
// of T4096 took 1.4 times as long as whole.  Backward: 8 of T256 63 / 37, of T4096 910 / 94; 64 of T256 65 / 48, of T4096 987 / 458; 128 of T256 66 / 65, of
// T4096 1010 / 780.  fp32 mode, forward: 64 of T256 43 / 41, 128 of T1024 158 / 178, of T4096 723 / 674; backward: 128 of T256 70 / 70, of T4096 997 / 863.
constexpr int BLOCK_CHUNKS = 4, SLOTS_FWD = 512, SLOTS_BWD = 256;
int time_blocks(int heads, int T, bool bwd, int* per) {
    const int want = (bwd ? SLOTS_BWD : SLOTS_FWD) / heads, nch = T / CL;
    *per = nch;
    if (want < (bwd ? 2 : 4) || nch < 4 * BLOCK_CHUNKS || (!bwd && nch * 16384LL < static_cast<long long>(heads) * heads * heads)) return 1;
    const int least = (nch + want - 1) / want;
    *per = least > BLOCK_CHUNKS ? least : BLOCK_CHUNKS;
    return (nch + *per - 1) / *per;
}
// Heads done as whole sequences, then others in NB blocks of `per` chunks.  More heads than CUs leave a last round of few workgroups, as long
// as the others: the heads beyond a multiple of the CUs are done in blocks where they are so few that this is shorter.  In the
// forward, where two workgroups of a CU get little more done than one, that is less to gain.  T1024, us whole / split, bf16 and fp32 mode,
// backward: 264 heads 497 / 316 and 513 / 355, 288 504 / 355 and 525 / 404, 320 532 / 419 and 530 / 459, 352 510 / 470 and 533 / 516, 384 527 / 490 and
// 541 / 547, 528 753 / 598 and 798 / 678, 576 779 / 681 and 814 / 771; forward: 264 236 / 200 and 274 / 247, 288 249 / 245 and 289 / 292, 320 270 / 295 and
// 296 / 334, 528 391 / 344 and 464 / 399, 576 401 / 404 and 496 / 481.  T256, backward: 264 134 / 105 and 138 / 117, 320 132 / 119 and 144 / 136, 352 136 / 136
// and 146 / 151; forward: 264 70 / 73 and 66 / 76, 528 97 / 100 and 104 / 121; T512, forward: 264 128 / 113 and 126 / 129.
// Errors of heads in 8 to 16 blocks against 64 bits, T1024, fp32 mode, 1e-7, whole -> in blocks: w = 0.5 the same; w = -8, where a state lasts, sT
// 1.04 -> 1.28 to 1.63, dk 1.27 -> 1.46 to 1.89; dw 21 -> 5 to 11 and 6.7 -> 3.7 to 4.4.
struct Split7 { int whole, rest, NB, per; };
constexpr int REST_FWD = 16, REST_FWD_CHUNKS = 48, REST_BWD = 96;
Split7 split_heads(int B, int T, int H, bool bwd) {
    if (static_cast<long long>(B) * H > 0x7fffffffLL) return {0, 0, 1, T / CL};      // (no memory holds them)
    const int all = B * H, rest = all % SLOTS_BWD;
    Split7 x{all - rest, rest, 1, T / CL};
    if (rest > 0 && (all < SLOTS_BWD || (bwd ? rest <= REST_BWD && T / CL * 4 >= rest : rest <= REST_FWD && T / CL >= REST_FWD_CHUNKS))) x.NB = time_blocks(rest, T, bwd, &x.per);
    return x.NB > 1 ? x : Split7{all, 0, 1, T / CL};
}
size_t blocks_bytes(size_t bh, int NB) { return NB > 1 ? bh * (NB - 1) * 3 * N * N * sizeof(float) + (bh * sizeof(int) + 15) / 16 * 16 : 0; }
// the kernels that bring the states to the borders of the blocks of the heads from p.at on
template <bool F32, bool REV> int cut(hipStream_t st, int heads, Args7c& p, void* ws) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(rwkv7c_local<F32, REV>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       static_cast<int>(L_TOTAL<F32>));
    if (attr != hipSuccess) { g_last_hip_error = static_cast<int>(attr); return RWKV_ERR_LAUNCH; }
    const size_t n = static_cast<size_t>(heads) * (p.NB - 1) * N * N;
    p.local = static_cast<float*>(ws); p.enter = p.local + 2 * n; p.flags = reinterpret_cast<int*>(p.enter + n);
    rwkv7c_local<F32, REV><<<dim3(heads, 1, 2 * (p.NB - 1)), dim3(NTF), L_TOTAL<F32>, st>>>(p);
    rwkv7c_scan<REV><<<dim3(4 * heads), dim3(256), 0, st>>>(p);
    return launch_status();
}
// whole sequences, then those in blocks: a launch each, of the heads from p.at on.  More than LAUNCH_HEADS are several: beyond 2^32 work items along
// x a launch does the remainder only, and reports no error (forward, 16 tokens of 8.4 million heads).
constexpr int LAUNCH_HEADS = 1 << 22;
static_assert(static_cast<long long>(LAUNCH_HEADS) * NTB < 1LL << 32 && LAUNCH_HEADS * static_cast<long long>(NTF) < 1LL << 32, "work items of a launch");
template <bool F32, bool REV, typename Whole, typename Blocks> int in_parts(hipStream_t st, int B, Args7c& p, void* ws, Whole whole, Blocks blocks) {
    Split7 x = split_heads(B, p.T, p.H, REV);
    if (x.whole + x.rest == 0) return RWKV_ERR_SHAPE;
    if (ws == nullptr) x = {B * p.H, 0, 1, p.T / CL};
    p.NB = 1; p.at = 0;
    for (; p.at < x.whole; p.at += LAUNCH_HEADS) {
        whole(p, dim3(std::min(x.whole - p.at, LAUNCH_HEADS)));
        if (int e = launch_status()) return e;
        if (x.whole - p.at <= LAUNCH_HEADS) break;           // (p.at would go beyond what an int holds)
    }
    if (x.rest == 0) return RWKV_OK;
    p.NB = x.NB; p.per = x.per; p.at = x.whole;
    if (int e = cut<F32, REV>(st, x.rest, p, ws)) return e;
    blocks(p, dim3(x.rest, 1, x.NB));
    return launch_status();
}

hipError_t raise_lds(void (*kernel)(Args7c), size_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
}
template <bool F32, bool KEEP> int start_fwd(hipStream_t st, int B, Args7c& p, void* ws) {
    static const hipError_t attr[2] = {raise_lds(rwkv7c_fwd<F32, KEEP, false>, F_TOTAL<F32>), raise_lds(rwkv7c_fwd<F32, KEEP, true>, F_TOTAL<F32>)};
    for (const hipError_t e : attr) if (e != hipSuccess) { g_last_hip_error = static_cast<int>(e); return RWKV_ERR_LAUNCH; }
    return in_parts<F32, false>(st, B, p, ws,
        [&](const Args7c& q, dim3 grid) { hipLaunchKernelGGL((rwkv7c_fwd<F32, KEEP, false>), grid, dim3(NTF), F_TOTAL<F32>, st, q); },
        [&](const Args7c& q, dim3 grid) { hipLaunchKernelGGL((rwkv7c_fwd<F32, KEEP, true>), grid, dim3(NTF), F_TOTAL<F32>, st, q); });
}
template <bool F32> int start_bwd(hipStream_t st, int B, Args7c& p, void* ws) {
    static_assert(LB<F32>::BYTES <= 160 * 1024, "the backward's LDS must fit one CU");
    static const hipError_t attr[2] = {raise_lds(rwkv7c_bwd<F32, false>, LB<F32>::BYTES), raise_lds(rwkv7c_bwd<F32, true>, LB<F32>::BYTES)};
    for (const hipError_t e : attr) if (e != hipSuccess) { g_last_hip_error = static_cast<int>(e); return RWKV_ERR_LAUNCH; }
    return in_parts<F32, true>(st, B, p, ws,
        [&](const Args7c& q, dim3 grid) { hipLaunchKernelGGL((rwkv7c_bwd<F32, false>), grid, dim3(NTB), LB<F32>::BYTES, st, q); },
        [&](const Args7c& q, dim3 grid) { hipLaunchKernelGGL((rwkv7c_bwd<F32, true>), grid, dim3(NTB), LB<F32>::BYTES, st, q); });
}

}  // namespace

size_t rwkv7c_workspace_bytes(int B, int T, int H, bool bwd) {
    const Split7 x = split_heads(B, T, H, bwd);
    return blocks_bytes(x.rest, x.NB);
}
int launch7c_fwd(hipStream_t st, bool f32, int B, int T, int H, const float* s0, const void* r, const void* w, const void* k,
                 const void* v, const void* a, const void* b, void* y, float* sT, float* s, float* sa, void* ws) {
    Args7c p{};
    p.T = T; p.H = H; p.s0 = s0; p.r = el(r); p.w = el(w); p.k = el(k); p.v = el(v); p.a = el(a); p.b = el(b); p.y = el(y);
    p.sT = sT; p.s = s; p.sa = sa;
    if (s != nullptr) return f32 ? start_fwd<true, true>(st, B, p, ws) : start_fwd<false, true>(st, B, p, ws);
    return f32 ? start_fwd<true, false>(st, B, p, ws) : start_fwd<false, false>(st, B, p, ws);
}

int launch7c_bwd(hipStream_t st, bool f32, int B, int T, int H, const void* r, const void* w, const void* k, const void* v,
                 const void* a, const void* b, const void* dy, const float* dsT, const float* s, const float* sa,
                 float* ds0, void* dr, void* dw, void* dk, void* dv, void* da, void* db, void* ws) {
    Args7c p{};
    p.T = T; p.H = H; p.r = el(r); p.w = el(w); p.k = el(k); p.v = el(v); p.a = el(a); p.b = el(b); p.dy = el(dy); p.dsT = dsT;
    p.s = const_cast<float*>(s); p.sa = const_cast<float*>(sa); p.ds0 = ds0;
    p.dr = el(dr); p.dw = el(dw); p.dk = el(dk); p.dv = el(dv); p.da = el(da); p.db = el(db);
    return f32 ? start_bwd<true>(st, B, p, ws) : start_bwd<false>(st, B, p, ws);
}

}  // namespace rwkv
