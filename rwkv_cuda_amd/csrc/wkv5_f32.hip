// wkv5 and wkv5a, fp32 I/O, head size 64, in CHUNKED form on the fp32 matrix cores (gfx950, v_mfma_f32_16x16x4_f32).
//
// Step form (wkv5/run.py:231-262, wkv5a/run.py:260-289), one head, S[i][j] (i value channel, j key channel):
//     y_t[i] = sum_j r_t[j] (S_t[i][j] + (u1[j] + u2[i]) k_t[j] v_t[i])       S_{t+1} = S_t o W + v_t k_t^T
// with W[i][j] = e^{l1[j] + l2[i]}, l = -exp(w_raw); wkv5 has l2 = 0 and u2 = 0 (TWO = false).  The decays are constant in
// time, so a power that a token of a chunk (L = 16 tokens, local t = 0..15) needs is the same in every chunk: all of them are
// made once per workgroup and live in registers, each exact to fp32 rounding.  S0 is the state entering the chunk, D the
// gradient of the state leaving it; o1 = e^{l1}, o2 = e^{l2}; m a reference token (8, the middle, unless the decay is strong):
//     A[t][s]  = sum_j (r_t o1^{t-m}) (k_s o1^{m-1-s})     B[t][s] = sum_i (gy_t o2^{t-m}) (v_s o2^{m-1-s})          s < t
//     y_t   = o2^t (r_t o1^t) S0^T        + o2^{t-m} sum_s A[t][s] (v_s o2^{m-1-s})      + bonus
//     dr_t  = o1^t (gy_t o2^t) S0         + o1^{t-m} sum_s B[t][s] (k_s o1^{m-1-s})      + bonus
//     dk_t  = o1^{15-t} (v_t o2^{15-t}) D + o1^{m-1-t} sum_s B[s][t] (r_s o1^{s-m})      + bonus
//     dv_t  = o2^{15-t} (k_t o1^{15-t}) D^T + o2^{m-1-t} sum_s A[s][t] (gy_s o2^{s-m})   + bonus
//     S_L   = S0 o W^16 + sum_s (v_s o2^{15-s})(k_s o1^{15-s})^T         D_0 = D o W^16 + sum_t (gy_t o2^t)(r_t o1^t)^T
// Decay gradient: a term (source s, sink t) of the output carries e^{l (t-1-s)}, so d/dl1[j] counts, for every such pair,
// the tokens strictly between s and t.  Cut at the chunk borders that is a sum of four kinds of products without any
// cancellation (the difference form used under bf16 outputs loses a digit per decade of T, which fp32 outputs show):
//     both in the chunk      sum_t r_t o1^{t-m} sum_s (t-1-s) B[t][s] (k_s o1^{m-1-s})
//     source before, sink in sum_t t r_t dr_t(S0 part)                  source in, sink after  sum_s (15-s) k_s dk_s(D part)
//     source before, sink after  16 sum_i S0 o W^16 o D
// Two-sided, the last three are kept per state element (the two middle ones become products over the tokens) and summed
// over i for l1 and over j for l2 at the end.
//
// Strong decays: with one reference in the middle a factor reaches e^{8 |l|}; beyond l = -7 (LAM_STRONG) the tiles take a
// reference in the middle of each half (m = 4, 12) and a pair of tokens of different halves carries o1^8 in addition: a second
// product for that quadrant, with o1^4 on either side (o1^8 itself may underflow where the whole term is one).  Heads with a
// channel below l = -17, or one that is no number, are left to wkv5_steps_* (steps_head, common.h).
//
// Inputs that are no number, or infinite: a tile product multiplies what it leaves out by zero, which would carry them to up to 15
// tokens that they do not act on (earlier outputs, later gradients).  The waves that load note them (one multiply-add an element;
// wkv5 B8 T4096 C4096, forward + backward, 2.03 -> 2.04 ms), and a head that has any is marked by a NaN in the first element of
// each of its outputs, which wkv5_steps_* look at: they do it over, step by step.  (The mark costs no workspace and no entry
// point, and a head whose first output is a NaN by itself is merely done twice.)
//
// What bounds it.  Forward: HBM (B8 T4096 C4096: 2.9 GB in 0.61 ms; the sequential kernel took 1.3).  Backward: the fp32 matrix
// instruction, which occupies a SIMD's vector ALU for 32 clocks (99 of them per SIMD and chunk and some 230 vector
// instructions fill two thirds of its 1.42 ms; the three sequential sweeps took 4.1).  wkv5a: 0.67 + 1.85 ms, 6.2 before.
#include <stddef.h>

#include "common.h"

namespace rwkv {
namespace {

constexpr int N = 64;
constexpr int L = 16;
constexpr int PS = 68;               // row stride (floats) of a [token][channel] plane
constexpr int TS = 20;               // row stride (floats) of a 16 x 16 tile
constexpr int NT = 512;              // forward: waves 0..3 products, 4..7 loads
constexpr int NTB = 512;             // backward: waves 0..3 D, 4..7 E
constexpr float LAM_STRONG = -7.f;

typedef float f32x4 __attribute__((ext_vector_type(4)));
DEVINL f32x4 mm(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
DEVINL f32x4 ld4(const float* p) { const float4 x = *reinterpret_cast<const float4*>(p); return f32x4{x.x, x.y, x.z, x.w}; }
DEVINL void st4(float* p, const f32x4& x) { *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]); }
constexpr f32x4 ZERO4 = {0.f, 0.f, 0.f, 0.f};
// four floats that need not sit in consecutive registers: for what a wave keeps across its loop (as vectors such values occupy
// aligned groups of four, and the register allocator spills and reloads whole groups for one of them)
struct F4 {
    float a[4];
    DEVINL float& operator[](int i) { return a[i]; }
    DEVINL float operator[](int i) const { return a[i]; }
};
DEVINL f32x4 operator*(const f32x4& x, const F4& y) { return f32x4{x[0] * y[0], x[1] * y[1], x[2] * y[2], x[3] * y[3]}; }
DEVINL f32x4 operator*(const F4& y, const f32x4& x) { return x * y; }

// states are saved for the backward at the start of every SEG-th chunk; the backward holds the states of a whole segment in
// registers and two segments' inputs in LDS: 3 chunks one-sided (150 of 160 KB), 2 with the two more planes of the other
template <bool TWO> constexpr int SEG = TWO ? 2 : 3;

struct ArgsC {
    int T, C, H;
    const float *r, *k, *v, *gy, *w, *u, *w2, *u2;      // w, w2 raw
    float *y, *gr, *gk, *gv;
    float *gw, *gu, *gw2, *gu2;                         // per-batch rows [B][C]
    float* saved;                                       // [B*H][segments][i][j]
    // sequences cut into blocks of time (NB > 1): blocks of `per` segments, a workgroup each; what each block leaves of a state that
    // entered it empty, [B*H][NB - 1][64][64] (the last block's is not needed, in the backward the first's); heads for the step kernels
    int B, NB, per;
    float* local;
    int* flags;
};

// Whole sequences (CUT = false) have an instance of their kernels of their own: with the choice left to run time what belongs to the
// blocks takes scalar and vector registers from them (B8 T4096 C4096 2.04 -> 2.02 ms).
template <bool CUT> DEVINL ArgsC only_whole(ArgsC p) {
    if constexpr (!CUT) p.NB = 1;
    return p;
}
// The workgroup's head and its part of the sequence: chunks first .. first + chunks - 1, tokens that are left from there on.
template <bool TWO> struct Part {
    int h, b, n, first, chunks, left;
    size_t bh, base;
};
template <bool TWO> DEVINL Part<TWO> part_of(const ArgsC& p) {
    Part<TWO> x;
    const int BH = p.B * p.H, nch = (p.T + L - 1) / L;
    // (divisions are done in vector registers)
    x.n = __builtin_amdgcn_readfirstlane(p.NB > 1 ? static_cast<int>(blockIdx.x) / BH : 0);
    x.bh = blockIdx.x - x.n * BH;
    x.b = __builtin_amdgcn_readfirstlane(static_cast<int>(x.bh) / p.H); x.h = static_cast<int>(x.bh) - x.b * p.H;
    x.first = x.n * p.per * SEG<TWO>;
    x.chunks = p.NB > 1 ? min(p.per * SEG<TWO>, nch - x.first) : nch;
    x.left = p.T - x.first * L;
    x.base = (static_cast<size_t>(x.b) * p.T + static_cast<size_t>(x.first) * L) * p.C + static_cast<size_t>(x.h) * N;
    return x;
}

// e^{lam n} for a small integer n, exact to fp32 rounding: the product and the base-2 exponent carry their rounding errors along
DEVINL float wpow(float lam, float n) {
    constexpr float L2E_HI = 1.44269502162933349609f, L2E_LO = 1.92596299112661746e-8f, LN2 = 0.69314718055994530942f;
    const float x = lam * n, lo = fmaf(lam, n, -x);
    const float t = x * L2E_HI;
    const float e = fmaf(x, L2E_HI, -t) + fmaf(x, L2E_LO, lo * L2E_HI);
    const float y = __builtin_amdgcn_exp2f(t);
    float r = fmaf(y, e * LN2, y);
    asm volatile("" : "+v"(r));        // (a scalar of its own: the compiler packs neighbouring powers into vectors otherwise)
    return r;
}
template <int R> DEVINL float row_ror(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + R, 0xf, 0xf, true));
}
// sum over the 16 lanes of a row, in all of them
DEVINL float row_sum(float x) {
    x += row_ror<8>(x); x += row_ror<4>(x); x += row_ror<2>(x); x += row_ror<1>(x);
    return x;
}

// The lane's number, worked out where it is used: what is derived from threadIdx is kept in registers, or spilled, across a loop.
DEVINL uint32_t lane_now() {
    uint32_t all = ~0u;
    asm volatile("" : "+s"(all));
    return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u));
}

struct Head { float lam[N], lam2[N], u[N], u2[N], dec[N], dec2[N], blk[N], blk2[N]; };      // decays of a chunk, of a block of time

// whether any element is no number, or infinite
DEVINL bool not_finite(const f32x4& a, const f32x4& b, const f32x4& c, const f32x4& d = ZERO4) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(a[e], 0.f, fmaf(b[e], 0.f, fmaf(c[e], 0.f, fmaf(d[e], 0.f, s))));
    return s != 0.f;
}
// the mark, by the lane that has written this element before; in blocks of time a word of the head's own, as other workgroups write that
DEVINL void mark(float* first) { *first = __builtin_nanf(""); }

// the head's parameters into LDS (by the first wave); every wave finds out for itself whether a decay is strong
template <bool TWO> DEVINL bool head_setup(Head& hd, const ArgsC& p, int h, int tid) {
    const int lane = tid & 63, c = h * N + lane;
    const float l1 = -expf(p.w[c]), l2 = TWO ? -expf(p.w2[c]) : 0.f;
    float mn = fminf(l1, l2);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o, 64));
    if (tid < N) {
        hd.lam[lane] = l1; hd.dec[lane] = wpow(l1, L); hd.u[lane] = p.u[c];
        hd.lam2[lane] = l2; hd.dec2[lane] = wpow(l2, L); hd.u2[lane] = TWO ? p.u2[c] : 0.f;
        const float len = static_cast<float>(p.per * SEG<TWO> * L);
        hd.blk[lane] = wpow(l1, len); hd.blk2[lane] = wpow(l2, len);
    }
    return __builtin_amdgcn_readfirstlane(mn < LAM_STRONG ? 1 : 0) != 0;
}
// reference token of token t
template <bool STRONG> DEVINL int ref(int t) { return STRONG ? (t < 8 ? 4 : 12) : 8; }

// the powers half_tile takes for a side with log decays lam
template <bool STRONG> DEVINL void tile_powers(const float* lam, int cb0, int l16, int g, F4 (&cx)[2], F4 (&cy)[2], F4 (&w4)[2]) {
    const int m = ref<STRONG>(l16);
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float l = lam[16 * (cb0 + z) + 4 * g + v];
            cx[z][v] = wpow(l, static_cast<float>(l16 - m));
            cy[z][v] = wpow(l, static_cast<float>(m - 1 - l16));
            w4[z][v] = wpow(l, 4.f);
        }
}
// A tile applied to four token rows: sum over slots (token 4 g + v) of a[v] b[v], where pairs of tokens of different halves of a
// strong chunk take the factor w4 of the output's lane twice; cross: this lane's operand row pairs with the other half.
template <bool STRONG> DEVINL f32x4 apply(const f32x4& a, const f32x4& b, bool cross, float w4) {
    f32x4 d = ZERO4;
    if constexpr (STRONG) {
        f32x4 o = ZERO4;
#pragma unroll
        for (int v = 0; v < 4; ++v) { d = mm(cross ? 0.f : a[v], b[v], d); o = mm(cross ? a[v] : 0.f, b[v], o); }
        return d + o * w4 * w4;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) d = mm(a[v], b[v], d);
    return d;
}

// four token rows (token 4 g + v) of an output; left: rows from this lane's first on that exist; whole: all of the chunk's do
DEVINL void store_rows(float* out, int lo, int C, int left, bool whole, const f32x4& x) {
    if (whole) {
#pragma unroll
        for (int v = 0; v < 4; ++v) (out + static_cast<size_t>(v) * C)[lo] = x[v];
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (v < left) (out + static_cast<size_t>(v) * C)[lo] = x[v];
    }
}

// where the states of the part's segments are
template <bool TWO> DEVINL float* saved_state(const ArgsC& p, const Part<TWO>& x) {
    const size_t nch = (p.T + L - 1) / L, nseg = (nch + SEG<TWO> - 1) / SEG<TWO>;
    return p.saved + (x.bh * nseg + x.first / SEG<TWO>) * N * N;
}

// step(the lane's sixteen elements of a block's state) for n blocks' states, `next` floats apart; four are under way at once
template <class F> DEVINL void add_up(const float* x, int next, int n, const F& step) {
    f32x4 y[4][4];
    int m = 0;
    for (; m + 4 <= n; m += 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i, x += next)
#pragma unroll
            for (int t = 0; t < 4; ++t) y[i][t] = ld4(x + 16 * t);
#pragma unroll
        for (int i = 0; i < 4; ++i) step(y[i]);
    }
#pragma unroll 1
    for (; m < n; ++m, x += next) {
#pragma unroll
        for (int t = 0; t < 4; ++t) y[0][t] = ld4(x + 16 * t);
        step(y[0]);
    }
}

// ---------------------------------------------------------------------------------------------------- blocks of time, first pass
// What a block leaves of an empty state: sum over its tokens of v_t k_t^T with the decay that is left to the block's end, or (REV) from
// the end backwards what the gradient state takes up, gy_t r_t^T.  Both are E[outer][inner] = sum_t Y_t[outer] X_t[inner] o^{15 - t} in
// chunks whose tokens are counted in the direction of travel; forward X = k, Y = v, backward X = gy, Y = r, so that a lane holds the
// element order of the state in the kernels that follow.  A workgroup makes 16 of the 64 outer channels, its waves a quarter of the
// block each, added up at the end.  Operands come from memory as the matrix instruction takes them.
template <bool TWO, bool REV>
__global__ __launch_bounds__(256) void wkv5c_local(const ArgsC p) {
    __shared__ f32x4 part[4][4][64];
    const int tid = threadIdx.x, lane = tid & 63, z = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int q = blockIdx.x & 3, BH = p.B * p.H, m = (blockIdx.x >> 2) / BH, bh = (blockIdx.x >> 2) - m * BH, b = bh / p.H, h = bh - b * p.H, C = p.C;
    const bool steps = steps_head<true, N>(p.w, TWO ? p.w2 : nullptr, h * N);
    if (m == 0 && q == 0 && tid == 0) p.flags[bh] = steps;
    if (steps) return;
    const float* const wx = REV ? (TWO ? p.w2 : nullptr) : p.w;
    const float* const wy = REV ? p.w : (TWO ? p.w2 : nullptr);
    const int n = REV ? m + 1 : m, nch = (p.T + L - 1) / L, first = n * p.per * SEG<TWO>, chunks = min(p.per * SEG<TWO>, nch - first), per = (chunks + 3) / 4;
    auto log_decay = [&](const float* w, int c) __attribute__((always_inline)) { return w != nullptr ? -expf(w[h * N + c]) : 0.f; };
    const int own = 16 * q + l16;
    const float ly = log_decay(wy, own), dy = wpow(ly, L);
    float px[4][4], py[4];                               // token 4 s + g, inner channel 16 t + l16
    F4 dx[4];                                            // o^16 of inner channel 16 t + 4 g + v
    float lx[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const float l = log_decay(wx, 16 * t + l16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            px[t][e] = wpow(l, static_cast<float>(15 - 4 * e - g));
            lx[t][e] = log_decay(wx, 16 * t + 4 * g + e);
            dx[t][e] = wpow(lx[t][e], L) * dy;
        }
        py[t] = wpow(ly, static_cast<float>(15 - 4 * t - g));
    }
    const float* const X = (REV ? p.gy : p.k) + static_cast<size_t>(b) * p.T * C + h * N;
    const float* const Y = (REV ? p.r : p.v) + static_cast<size_t>(b) * p.T * C + h * N;
    const int c0 = min(z * per, chunks), c1 = min(c0 + per, chunks);        // counted in the direction of travel
    struct Rows { float x[4][4], y[4]; };
    auto fetch = [&](const int i, Rows& d) __attribute__((always_inline)) {
        const int c = first + (REV ? chunks - 1 - min(i, chunks - 1) : min(i, chunks - 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = c * L + (REV ? 15 - 4 * e - g : 4 * e + g);
            const size_t o = static_cast<size_t>(min(t, p.T - 1)) * C;
            const bool in = t < p.T;
#pragma unroll
            for (int k = 0; k < 4; ++k) { const float x = X[o + 16 * k + l16]; d.x[k][e] = in ? x : 0.f; }
            const float y = Y[o + own];
            d.y[e] = in ? y : 0.f;
        }
    };
    f32x4 acc[4] = {ZERO4, ZERO4, ZERO4, ZERO4};
    Rows now, next;
    fetch(c0, now);
    for (int i = c0; i < c1; ++i) {
        fetch(i + 1, next);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 a = acc[t] * dx[t];
#pragma unroll
            for (int e = 0; e < 4; ++e) a = mm(now.x[t][e] * px[t][e], now.y[e] * py[e], a);
            acc[t] = a;
        }
        now = next;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) part[z][t][lane] = acc[t];
    __syncthreads();
    f32x4 s = part[0][z][lane];                          // inner channels 16 z + 4 g + v
#pragma unroll
    for (int i = 1; i < 4; ++i) {
        const float len = static_cast<float>(L * (min((i + 1) * per, chunks) - min(i * per, chunks)));
        f32x4 e;
#pragma unroll
        for (int v = 0; v < 4; ++v) e[v] = wpow(z == 0 ? lx[0][v] : (z == 1 ? lx[1][v] : (z == 2 ? lx[2][v] : lx[3][v])), len) * wpow(ly, len);
        s = s * e + part[i][z][lane];
    }
    st4(p.local + (static_cast<size_t>(bh) * (p.NB - 1) + m) * N * N + own * N + 16 * z + 4 * g, s);
}

// ---------------------------------------------------------------------------------------------------- forward
// Waves 0..3 (value channels 16 q + l16): St[jt][v] = S[i = 16 q + l16][j = 16 jt + 4 g + v], as it stands the B operand of a
// contraction over j.  Waves 4..7 load: chunk c + 2 into LDS while chunk c is worked on (three slots, one barrier a chunk),
// their global loads four chunks further ahead.  Wave q makes a quarter of the next chunk's tile (16 of the 64 key channels).
struct SlotF {
    float r[L][PS], k[L][PS], v[L][PS];
    float ruk[L], rk[L];
};
struct SmemF {
    Head hd;
    SlotF slot[3];
    float part[2][4][L][TS];            // the four waves' parts of the tile, of this chunk and the next
    int marked;
};
constexpr int FDEPTH = 4;

template <bool TWO, bool STRONG, bool CUT>
DEVINL void fwd_products(SmemF& S, const ArgsC& p, int q, int lane, const Part<TWO>& part) {
    const int l16 = lane & 15, g = lane >> 4, T = part.left, C = p.C, nch = part.chunks;
    const size_t base = part.base;
    const int own = 16 * q + l16;
    f32x4 St[4] = {ZERO4, ZERO4, ZERO4, ZERO4};
    if (part.n > 0) {                                    // the state that enters the block, from what the blocks before leave
        const float* x = p.local + part.bh * (p.NB - 1) * N * N + own * N + 4 * g;
        const float e2 = TWO ? S.hd.blk2[own] : 1.f;
        auto step = [&](const f32x4 (&y)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) St[jt] = St[jt] * (ld4(&S.hd.blk[16 * jt + 4 * g]) * e2) + y[jt];
        };
        add_up(x, N * N, part.n, step);
    }
    __builtin_amdgcn_sched_barrier(0);
    // powers: A operands over j (r o1^t, token t = l16; k o1^{15-t}, token 4 g + v), the tile's, the value side's
    F4 crs[4], cke[4], ctx, cty, ct4;
    {
        const int m = ref<STRONG>(l16);
#pragma unroll
        for (int jt = 0; jt < 4; ++jt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                crs[jt][v] = wpow(S.hd.lam[16 * jt + 4 * g + v], static_cast<float>(l16));
                cke[jt][v] = wpow(S.hd.lam[16 * jt + l16], static_cast<float>(15 - 4 * g - v));
            }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float l = S.hd.lam[16 * q + 4 * g + v];
            ctx[v] = wpow(l, static_cast<float>(l16 - m));
            cty[v] = wpow(l, static_cast<float>(m - 1 - l16));
            ct4[v] = wpow(l, 4.f);
        }
    }
    F4 c2s = {}, c2m = {}, c2k = {}, c2e = {};
    float u2 = 0.f, d2 = 1.f, w24 = 1.f;
    if constexpr (TWO) {
        const float l = S.hd.lam2[own];
        u2 = S.hd.u2[own];
        if constexpr (!CUT) { d2 = S.hd.dec2[own]; w24 = wpow(l, 4.f); }       // (with blocks of time anew in every chunk: the registers do not reach)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 4 * g + v, m = ref<STRONG>(t);
            c2s[v] = wpow(l, static_cast<float>(t)); c2e[v] = wpow(l, static_cast<float>(15 - t));
            c2m[v] = wpow(l, static_cast<float>(t - m)); c2k[v] = wpow(l, static_cast<float>(m - 1 - t));
        }
    }
    auto tile = [&](const SlotF& s, float (*out)[TS]) __attribute__((always_inline)) {
        const f32x4 xa = ld4(&s.r[l16][16 * q + 4 * g]) * ctx, ya = ld4(&s.k[l16][16 * q + 4 * g]) * cty;
        f32x4 acc = ZERO4;
#pragma unroll
        for (int v = 0; v < 4; ++v) acc = mm(xa[v], ya[v], acc);
        if constexpr (STRONG) {
            f32x4 o = ZERO4;
#pragma unroll
            for (int v = 0; v < 4; ++v) o = mm(xa[v] * ct4[v], ya[v] * ct4[v], o);
            if (g >= 2 && l16 < 8) acc = o;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) out[4 * g + v][l16] = l16 < 4 * g + v ? acc[v] : 0.f;
    };
    float* const sv = p.saved != nullptr ? saved_state<TWO>(p, part) : nullptr;
    __syncthreads();                                     // chunks 0 and 1 are there
    tile(S.slot[0], S.part[0][q]);
    __syncthreads();
    int sl = 0;
    const int lo = 4 * g * C + own;
    for (int c = 0; c < nch; ++c) {
        const SlotF& X = S.slot[sl];
        sl = sl == 2 ? 0 : sl + 1;
        if (c + 1 < nch) tile(S.slot[sl], S.part[(c + 1) & 1][q]);
        if (sv != nullptr && (c > 0 || part.n > 0) && c % SEG<TWO> == 0) {
            char* d = reinterpret_cast<char*>(sv + static_cast<size_t>(c / SEG<TWO>) * N * N);
            const uint32_t me = lane_now(), so = ((16 * q + (me & 15)) * N + 4 * (me >> 4)) * 4;
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) st4(reinterpret_cast<float*>(d + 64 * jt + so), St[jt]);
        }
        f32x4 y2[2] = {ZERO4, ZERO4};
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
            const f32x4 xa = ld4(&X.r[l16][16 * jt + 4 * g]) * crs[jt];
#pragma unroll
            for (int v = 0; v < 4; ++v) y2[jt & 1] = mm(xa[v], St[jt][v], y2[jt & 1]);
        }
        f32x4 vop;                                       // v[token 4 g + v][own]
#pragma unroll
        for (int v = 0; v < 4; ++v) vop[v] = X.v[4 * g + v][own];
        const float (*pt)[L][TS] = S.part[c & 1];
        const f32x4 at = (ld4(&pt[0][l16][4 * g]) + ld4(&pt[1][l16][4 * g])) + (ld4(&pt[2][l16][4 * g]) + ld4(&pt[3][l16][4 * g]));
        const f32x4 ruk = ld4(&X.ruk[4 * g]);
        f32x4 y = y2[0] + y2[1];
        if constexpr (TWO) {
            const f32x4 ap = apply<STRONG>(at, vop * c2k, l16 >= 8 && g < 2, STRONG && CUT ? wpow(S.hd.lam2[own], 4.f) : w24);
            y = y * c2s + ap * c2m + vop * (ruk + u2 * ld4(&X.rk[4 * g]));
        } else {
            y += vop * ruk;
#pragma unroll
            for (int v = 0; v < 4; ++v) y = mm(at[v], vop[v], y);
        }
        float* const out = p.y + base + static_cast<size_t>(c) * L * C;
        store_rows(out, lo, C, T - c * L - 4 * g, c * L + L <= T, y);
        const f32x4 ve = TWO ? vop * c2e : vop;
        if constexpr (TWO && CUT) d2 = S.hd.dec2[own];
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
            f32x4 acc = St[jt] * ld4(&S.hd.dec[16 * jt + 4 * g]);
            if constexpr (TWO) acc *= d2;
#pragma unroll
            for (int v = 0; v < 4; ++v) acc = mm(X.k[4 * g + v][16 * jt + l16] * cke[jt][v], ve[v], acc);
            St[jt] = acc;
        }
        __syncthreads();
    }
    if (q == 0 && lane == 0 && S.marked) { if (p.NB > 1) p.flags[part.bh] = 1; else mark(p.y + base); }
}

template <bool TWO, bool CUT>
__global__ __launch_bounds__(NT, 4) void wkv5c_fwd(const ArgsC args) {
    const ArgsC p = only_whole<CUT>(args);
    __shared__ SmemF S;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), q = w & 3;
    const Part<TWO> part = part_of<TWO>(p);
    const int h = part.h, T = part.left, C = p.C, nch = part.chunks;
    const size_t base = part.base;
    if (steps_head<true, N>(p.w, TWO ? p.w2 : nullptr, h * N)) return;
    const bool strong = head_setup<TWO>(S.hd, p, h, tid);
    if (tid == 0) S.marked = 0;
    __syncthreads();
    if (w >= 4) {
        const int tp = tid - 256, row = tp >> 4, c4 = (tp & 15) * 4;
        const f32x4 u = ld4(&S.hd.u[c4]);
        f32x4 x[FDEPTH][3];
        auto fetch = [&](const int c, f32x4 (&d)[3]) __attribute__((always_inline)) {
            const int cc = min(c, nch - 1);                       // (the same loads in every iteration: see the backward of wkv6)
            const size_t o = base + static_cast<size_t>(cc) * L * C;
            const int lo = min(row, T - 1 - cc * L) * C + c4;
            d[0] = ld4(p.r + o + lo); d[1] = ld4(p.k + o + lo); d[2] = ld4(p.v + o + lo);
        };
        auto put = [&](const int c, SlotF& s, const f32x4 (&d)[3]) __attribute__((always_inline)) {
            f32x4 r = d[0], k = d[1], v = d[2];
            if (c * L + L > T && c * L + row >= T) { r = ZERO4; k = ZERO4; v = ZERO4; }
            st4(&s.r[row][c4], r); st4(&s.k[row][c4], k); st4(&s.v[row][c4], v);
            if (not_finite(r, k, v)) S.marked = 1;
            const f32x4 rk = r * k;
            const float a = row_sum((rk[0] * u[0] + rk[1] * u[1]) + (rk[2] * u[2] + rk[3] * u[3]));
            if ((tp & 15) == 0) s.ruk[row] = a;
            if constexpr (TWO) {
                const float a2 = row_sum((rk[0] + rk[1]) + (rk[2] + rk[3]));
                if ((tp & 15) == 0) s.rk[row] = a2;
            }
        };
#pragma unroll
        for (int z = 0; z < FDEPTH; ++z) fetch(z, x[z]);
        put(0, S.slot[0], x[0]); fetch(FDEPTH, x[0]);
        put(1, S.slot[1], x[1]); fetch(FDEPTH + 1, x[1]);
        __syncthreads();
        __syncthreads();
        int sl = 2;
        for (int c0 = 0; c0 < nch; c0 += FDEPTH) {
#pragma unroll
            for (int z = 0; z < FDEPTH; ++z) {
                const int c = c0 + z;
                if (c >= nch) break;
                put(c + 2, S.slot[sl], x[(z + 2) % FDEPTH]);
                fetch(c + 2 + FDEPTH, x[(z + 2) % FDEPTH]);
                sl = sl == 2 ? 0 : sl + 1;
                __syncthreads();
            }
        }
        return;
    }
    if (strong) fwd_products<TWO, true, CUT>(S, p, q, lane, part);
    else fwd_products<TWO, false, CUT>(S, p, q, lane, part);
}

// ---------------------------------------------------------------------------------------------------- backward
// One reverse sweep, one barrier a chunk, eight waves, two roles of four:
//   D, waves 0..3 (key channel j = 16 q + l16): the states of a segment, rebuilt from the saved one, and the gradient state, both
//      as S[i = 16 ib + 4 g + v][j], the B operands of contractions over the value channel: gr, gk, gw, gu.  The gradient state
//      goes through LDS to the E waves, which take it transposed (a second copy with an update of its own: 14 % more matrix
//      instructions).
//   E, waves 4..7 (value channel i = 16 q + l16): gv; the halves of the next chunk's two tiles (two waves the A tile, two the B
//      tile); all loads, SEG chunks ahead of their use.
// (Three roles on twelve waves, S and D apart: 168 registers a wave did not hold them, and no faster without the spills.)
// The planes in LDS are the raw inputs (two-sided: two scaled ones in addition): a power is applied to an operand on its way
// into the matrix instruction, from registers, so that a chunk costs four planes instead of one per power.
template <bool TWO> struct SlotB {
    float r[L][PS], k[L][PS], v[L][PS], g[L][PS];
    float gs_[TWO ? L : 1][PS], ve_[TWO ? L : 1][PS];       // two-sided: gy o2^t, v o2^{15-t}, which would take 64 registers as powers
    float vg[L], u2vg[L], ruk[L], rk[L];
};
template <bool TWO> struct SmemB {
    Head hd;
    SlotB<TWO> slot[2 * SEG<TWO>];
    float part[2][4][L][TS];            // halves of the tiles A (0, 1) and B (2, 3)
    float ds[2][N][PS];                 // the gradient state of the chunk, for the E waves: [chunk parity][i][j]
    float red[TWO ? 4 : 1][N];          // two-sided: the waves' sums over j of the per-element gradient
    int marked;
};

// LDS by byte offset: the position of the chunk's slot (uniform) plus one of a few per-lane offsets, everything else an
// immediate of the instruction.  The sum is hidden from the optimiser once per chunk: left alone it keeps (lane offset + field)
// of every field in a register of its own across the loop, and spills them.
extern __shared__ __align__(16) unsigned char smem_raw[];
DEVINL f32x4 lds4(uint32_t o) { return *reinterpret_cast<const f32x4*>(smem_raw + o); }
DEVINL float lds1(uint32_t o) { return *reinterpret_cast<const float*>(smem_raw + o); }
DEVINL uint32_t hide(uint32_t o) { asm volatile("" : "+v"(o)); return o; }
constexpr uint32_t ROWB = PS * 4, TROWB = TS * 4, TILEB = L * TROWB;
// rows 4 g + v, v = 0..3, of one column
template <uint32_t STRIDE = ROWB> DEVINL f32x4 col4(uint32_t o) { return f32x4{lds1(o), lds1(o + STRIDE), lds1(o + 2 * STRIDE), lds1(o + 3 * STRIDE)}; }
template <bool TWO> struct At {                            // byte offsets within LDS and within a slot
    using M = SmemB<TWO>;
    using B = SlotB<TWO>;
    static constexpr uint32_t DEC2 = offsetof(M, hd) + offsetof(Head, dec2), PART = offsetof(M, part), DS = offsetof(M, ds), DSB = sizeof(M::ds) / 2;
    static constexpr uint32_t R = offsetof(B, r), K = offsetof(B, k), V = offsetof(B, v), GY = offsetof(B, g);
    static constexpr uint32_t GS = TWO ? offsetof(B, gs_) : GY, VE = TWO ? offsetof(B, ve_) : V;       // gy o2^t, v o2^{15-t}
    static constexpr uint32_t VG = offsetof(B, vg), U2VG = offsetof(B, u2vg), RUK = offsetof(B, ruk), RK = offsetof(B, rk);
    static DEVINL uint32_t slot(int c) { return offsetof(M, slot) + static_cast<uint32_t>(c % (2 * SEG<TWO>)) * sizeof(B); }
    static DEVINL uint32_t tile(int c, int half) { return PART + static_cast<uint32_t>((c & 1) * 4 + half) * TILEB; }
    static DEVINL uint32_t ds(int c) { return DS + static_cast<uint32_t>(c & 1) * DSB; }
};

// One half (32 channels, two 16-channel blocks) of a causal tile sum_c X[t][c] Y[s][c], s < t, from the plane rows at x and y to
// the tile column at out, with the powers cx (of t = l16) and cy (of s = l16) per channel block and register; w4: half of what
// pairs across the halves of a strong chunk carry.
template <bool SCALED, bool STRONG>
DEVINL void half_tile(uint32_t x, uint32_t y, uint32_t out, const F4 (&cx)[2], const F4 (&cy)[2], const F4 (&w4)[2], int l16, int g) {
    f32x4 d[2] = {ZERO4, ZERO4};
    f32x4 xa[2], ya[2];
#pragma unroll
    for (int z = 0; z < 2; ++z) {
        xa[z] = lds4(x + 64 * z); ya[z] = lds4(y + 64 * z);
        if constexpr (SCALED) { xa[z] = xa[z] * cx[z]; ya[z] = ya[z] * cy[z]; }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int z = 0; z < 2; ++z) d[z] = mm(xa[z][v], ya[z][v], d[z]);
    f32x4 acc = d[0] + d[1];
    if constexpr (SCALED && STRONG) {
        f32x4 o = ZERO4;
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int v = 0; v < 4; ++v) o = mm(xa[z][v] * w4[z][v], ya[z][v] * w4[z][v], o);
        if (g >= 2 && l16 < 8) acc = o;
    }
    // acc[v] = tile[t = 4 g + v][s = l16]
#pragma unroll
    for (int v = 0; v < 4; ++v) *reinterpret_cast<float*>(smem_raw + out + v * TROWB) = l16 < 4 * g + v ? acc[v] : 0.f;
}
// the gradient state from the D waves' layout, x[ib][v] = D[i = 16 ib + 4 g + v][j = own], to LDS as rows
DEVINL void hand_over(uint32_t o, const f32x4 (&x)[4]) {
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int v = 0; v < 4; ++v) *reinterpret_cast<float*>(smem_raw + o + (16 * ib + v) * ROWB) = x[ib][v];
}
DEVINL float sum4(const f32x4& x) { return (x[0] + x[1]) + (x[2] + x[3]); }
// two-sided: a lane's per-element sums acc[i = 16 ib + 4 g + v][j] summed over the wave's sixteen j
DEVINL void reduce_cols(float* red, const f32x4 (&acc)[4], int l16, int g) {
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float x = row_sum(acc[ib][v]);
            if (l16 == 0) red[16 * ib + 4 * g + v] = x;
        }
}
DEVINL void store_chunk(float* p, size_t base, int c, int g, int own, int C, int T, const f32x4& x) {
    store_rows(p + base + static_cast<size_t>(c) * L * C, 4 * g * C + own, C, T - c * L - 4 * g, c * L + L <= T, x);
}

template <bool TWO, bool STRONG>
DEVINL void role_d(SmemB<TWO>& S, const ArgsC& p, int q, int lane, const Part<TWO>& part) {
    constexpr int G = SEG<TWO>;
    using A = At<TWO>;
    const int l16 = lane & 15, g = lane >> 4, own = 16 * q + l16, C = p.C, T = part.left, nch = part.chunks;
    const size_t base = part.base;
    const bool later = part.n > 0;                       // a state enters the first segment
    const uint32_t orow = l16 * ROWB + 16 * g, ocol = 4 * g * ROWB + 4 * own, oall = 4 * g * ROWB + 4 * l16;      // [l16][4 g ..], [4 g + v][own], [4 g + v][l16]
    const uint32_t otr = l16 * TROWB + 16 * g, otc = 4 * g * TROWB + 4 * l16;
    const int nseg = (nch + G - 1) / G;
    const float* const sv = saved_state<TWO>(p, part) + 4 * g * N + own;
    const float l1 = S.hd.lam[own], u1 = S.hd.u[own], d1 = S.hd.dec[own], w4 = wpow(l1, 4.f);
    F4 cs, ce, cm, ck, tf, tr15, lag;                    // o1^t, o1^{15-t}, o1^{t-m}, o1^{m-1-t}, t, 15 - t for t = 4 g + v; t' - 1 - t for t' = l16
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int t = 4 * g + v, m = ref<STRONG>(t);
        tf[v] = static_cast<float>(t); tr15[v] = static_cast<float>(15 - t); lag[v] = static_cast<float>(l16 - 1 - t);
        cs[v] = wpow(l1, static_cast<float>(t)); ce[v] = wpow(l1, static_cast<float>(15 - t));
        cm[v] = wpow(l1, static_cast<float>(t - m)); ck[v] = wpow(l1, static_cast<float>(m - 1 - t));
    }
    f32x4 St[G][4], Sn[4], dS[4] = {ZERO4, ZERO4, ZERO4, ZERO4};
    f32x4 accG[TWO ? 4 : 1];
#pragma unroll
    for (int e = 0; e < (TWO ? 4 : 1); ++e) accG[e] = ZERO4;
    float gw = 0.f, gP = 0.f, gu = 0.f;
    auto fetch_state = [&](const int s) __attribute__((always_inline)) {
        const float* d = sv + static_cast<size_t>(max(s, 0)) * N * N;
#pragma unroll
        for (int ib = 0; ib < 4; ++ib)
#pragma unroll
            for (int v = 0; v < 4; ++v) Sn[ib][v] = s > 0 || later ? d[(16 * ib + v) * N] : 0.f;      // the sequence starts from nothing
    };
    auto decay = [&](const int ib) __attribute__((always_inline)) {
        if constexpr (TWO) return lds4(hide(16 * g) + A::DEC2 + 64 * ib) * d1;
        else return f32x4{d1, d1, d1, d1};
    };
    // rows of the value side for the next chunk, asked for before the barrier that ends this one (they have been there since
    // long ago; the first matrix instructions after a barrier would wait for all waves' reads at once)
    f32x4 gx[4], vx[4];
    auto rows = [&](const int c) __attribute__((always_inline)) {
        const uint32_t xr = hide(A::slot(max(c, 0)) + orow);
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) { gx[ib] = lds4(xr + A::GS + 64 * ib); vx[ib] = lds4(xr + A::VE + 64 * ib); }
    };
    auto chunk = [&](const int c, const f32x4 (&Sz)[4]) __attribute__((always_inline)) {
        const uint32_t sx = A::slot(c), xc = hide(sx + ocol), xd = hide(sx + oall), xg = hide(sx + 16 * g);
        const uint32_t tr = hide(A::tile(c, 2) + otr), tc = hide(A::tile(c, 2) + otc);
        f32x4 x2[2] = {ZERO4, ZERO4}, z2[2] = {ZERO4, ZERO4};
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                x2[ib & 1] = mm(gx[ib][v], Sz[ib][v], x2[ib & 1]);
                z2[ib & 1] = mm(vx[ib][v], dS[ib][v], z2[ib & 1]);
            }
        }
        const f32x4 kk = col4(xc + A::K), rr = col4(xc + A::R);
        const f32x4 rs = rr * cs;
        if constexpr (TWO) {
            const f32x4 rt = rs * tf, kt = kk * ce * tr15;
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) {
                const f32x4 ga = col4(xd + A::GS + 64 * ib), va = col4(xd + A::VE + 64 * ib), dec = decay(ib);
                f32x4 m1 = ZERO4, n1 = ZERO4, acc = dS[ib] * dec;
#pragma unroll
                for (int v = 0; v < 4; ++v) { m1 = mm(ga[v], rt[v], m1); n1 = mm(va[v], kt[v], n1); acc = mm(ga[v], rs[v], acc); }
                accG[ib] += Sz[ib] * (m1 + (16.f * dec) * dS[ib]) + dS[ib] * n1;
                dS[ib] = acc;
            }
        } else {
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) {
                const f32x4 ga = col4(xd + A::GS + 64 * ib);
                gP += sum4(Sz[ib] * dS[ib]);
                f32x4 acc = dS[ib] * d1;
#pragma unroll
                for (int v = 0; v < 4; ++v) acc = mm(ga[v], rs[v], acc);
                dS[ib] = acc;
            }
        }
        if (c > 0) hand_over(hide(A::ds(c - 1) + ocol), dS);
        if constexpr (!TWO) rows(c - 1);
        const f32x4 bm = lds4(tr) + lds4(tr + TILEB), bt = col4<TROWB>(tc) + col4<TROWB>(tc + TILEB);
        const f32x4 km = kk * ck, rm = rr * cm;
        const bool cx = l16 >= 8 && g < 2, cz = l16 < 8 && g >= 2;
        const f32x4 tx = apply<STRONG>(bm, km, cx, w4), tl = apply<STRONG>(bm * lag, km, cx, w4), tz = apply<STRONG>(bt, rm, cz, w4);
        const f32x4 xs = (x2[0] + x2[1]) * cs, zs = (z2[0] + z2[1]) * ce;
        const f32x4 vg = lds4(xg + A::VG);
        f32x4 bo = vg * u1;
        if constexpr (TWO) bo += lds4(xg + A::U2VG);
        gu += sum4(rr * kk * vg);
        gw += sum4(rm * tl);
        if constexpr (!TWO) gw += sum4(rr * xs * tf + kk * zs * tr15);
        store_chunk(p.gr, base, c, g, own, C, T, xs + tx * cm + kk * bo);
        store_chunk(p.gk, base, c, g, own, C, T, zs + tz * ck + rr * bo);
        if constexpr (TWO) rows(c - 1);                  // (earlier, under the products above, the registers do not reach for this)
    };
    fetch_state(nseg - 1);
    if (part.n + 1 < p.NB) {                             // the gradient of the state that leaves the block, from what the blocks after take up
        const float* x = p.local + (part.bh * (p.NB - 1) + p.NB - 2) * N * N + own * N + 4 * g;
        const float e1 = S.hd.blk[own];
        auto step = [&](const f32x4 (&y)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) dS[ib] = dS[ib] * (TWO ? ld4(&S.hd.blk2[16 * ib + 4 * g]) * e1 : f32x4{e1, e1, e1, e1}) + y[ib];
        };
        add_up(x, -N * N, p.NB - 1 - part.n, step);
    }
    hand_over(A::ds(nch - 1) + ocol, dS);
    __syncthreads();                                     // the top chunks are there
    rows(nch - 1);
    __syncthreads();                                     // and the first tiles
    for (int s = nseg - 1; s >= 0; --s) {
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) St[0][ib] = Sn[ib];
        fetch_state(s - 1);
#pragma unroll
        for (int z = 0; z + 1 < G; ++z) {
            if (s * G + z + 1 < nch) {
                const uint32_t sx = A::slot(s * G + z), xc = hide(sx + ocol), xd = hide(sx + oall);
                const f32x4 ke = col4(xc + A::K) * ce;
#pragma unroll
                for (int ib = 0; ib < 4; ++ib) {
                    const f32x4 va = col4(xd + A::VE + 64 * ib);
                    f32x4 acc = St[z][ib] * decay(ib);
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc = mm(va[v], ke[v], acc);
                    St[z + 1][ib] = acc;
                }
            }
        }
#pragma unroll
        for (int z = G - 1; z >= 0; --z) {
            const int c = s * G + z;
            if (c < nch) {
                chunk(c, St[z]);
                __syncthreads();
            }
        }
    }
    gw = fmaf(16.f * d1, gP, gw);
    if constexpr (TWO) {
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) gw += sum4(accG[ib]);
        reduce_cols(S.red[q], accG, l16, g);
    }
    __syncthreads();
    gw = allreduce_rows(gw); gu = allreduce_rows(gu);
    if (g == 0) {
        const size_t o = (static_cast<size_t>(part.n) * p.B + part.b) * C + part.h * N + own;
        p.gw[o] = l1 * gw;
        p.gu[o] = gu;
    }
    if (q == 0 && lane == 0 && S.marked) { if (p.NB > 1) p.flags[part.bh] = 1; else { mark(p.gr + base); mark(p.gk + base); } }
}

template <bool TWO, bool STRONG>
DEVINL void role_e(SmemB<TWO>& S, const ArgsC& p, int q, int lane, const Part<TWO>& part) {
    constexpr int G = SEG<TWO>;
    using A = At<TWO>;
    const int l16 = lane & 15, g = lane >> 4, own = 16 * q + l16, C = p.C, T = part.left, nch = part.chunks;
    const size_t base = part.base;
    const uint32_t orow = l16 * ROWB + 16 * g, ocol = 4 * g * ROWB + 4 * own;                // [l16][4 g ..], [4 g + v][own]
    const uint32_t otr = l16 * TROWB + 16 * g, otc = 4 * g * TROWB + 4 * l16, odt = own * ROWB + 16 * g;
    const int te = 64 * q + lane, row = te >> 4, c4 = (te & 15) * 4;
    // loads: chunk c - G is written in the phase of chunk c, out of registers that asked for it G phases before
    F4 u, u2c;
#pragma unroll
    for (int e = 0; e < 4; ++e) { u[e] = S.hd.u[c4 + e]; u2c[e] = S.hd.u2[c4 + e]; }
    F4 pgs = {}, pve = {};
    if constexpr (TWO) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            pgs[e] = wpow(S.hd.lam2[c4 + e], static_cast<float>(row));
            pve[e] = wpow(S.hd.lam2[c4 + e], static_cast<float>(15 - row));
        }
    }
    auto fetch = [&](const int c, f32x4 (&d)[4]) __attribute__((always_inline)) {
        const int cc = max(c, 0);
        const size_t o = base + static_cast<size_t>(cc) * L * C;
        const int lo = min(row, T - 1 - cc * L) * C + c4;
        d[0] = ld4(p.r + o + lo); d[1] = ld4(p.k + o + lo); d[2] = ld4(p.v + o + lo); d[3] = ld4(p.gy + o + lo);
    };
    auto put = [&](const int c, const f32x4 (&d)[4]) __attribute__((always_inline)) {
        SlotB<TWO>& s = S.slot[c % (2 * G)];
        f32x4 r = d[0], k = d[1], v = d[2], gy = d[3];
        if (c * L + L > T && c * L + row >= T) { r = ZERO4; k = ZERO4; v = ZERO4; gy = ZERO4; }
        st4(&s.r[row][c4], r); st4(&s.k[row][c4], k); st4(&s.v[row][c4], v); st4(&s.g[row][c4], gy);
        if (not_finite(r, k, v, gy)) S.marked = 1;
        if constexpr (TWO) { st4(&s.gs_[row][c4], gy * pgs); st4(&s.ve_[row][c4], v * pve); }
        const f32x4 rk = r * k, vg = v * gy;
        const float a = row_sum(sum4(rk * u)), e = row_sum(sum4(vg));
        if ((te & 15) == 0) { s.ruk[row] = a; s.vg[row] = e; }
        if constexpr (TWO) {
            const float a2 = row_sum(sum4(rk)), e2 = row_sum(sum4(vg * u2c));
            if ((te & 15) == 0) { s.rk[row] = a2; s.u2vg[row] = e2; }
        }
    };
    f32x4 ring[G][4];
    {
        f32x4 top[G][4];
#pragma unroll
        for (int z = 0; z < G; ++z) fetch(nch - 1 - z, top[z]);
#pragma unroll
        for (int z = 0; z < G; ++z)
            if (nch - 1 - z >= 0) put(nch - 1 - z, top[z]);
    }
    // the segment's position of chunk c - G is that of chunk c: its registers are ring[c % G]
    const int ctop = nch - 1 - (nch - 1) % G;            // first chunk of the top segment
#pragma unroll
    for (int z = 0; z < G; ++z) fetch(ctop + z < nch ? ctop + z - G : ctop + z - 2 * G, ring[z]);

    // powers: the A operand k o1^{15-t} (token l16); the tile half of this wave
    F4 cke[4], tx[2], ty[2], t4[2], lag;
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
#pragma unroll
        for (int v = 0; v < 4; ++v) cke[jt][v] = wpow(S.hd.lam[16 * jt + 4 * g + v], static_cast<float>(15 - l16));
    const int cb0 = 2 * (q & 1);
    tile_powers<STRONG>(q < 2 ? S.hd.lam : S.hd.lam2, cb0, l16, g, tx, ty, t4);
    auto tile = [&](const int c) __attribute__((always_inline)) {
        const uint32_t xr = hide(A::slot(c) + orow + 64 * cb0), out = hide(A::tile(c, q) + otc);
        if (q < 2) half_tile<true, STRONG>(xr + A::R, xr + A::K, out, tx, ty, t4, l16, g);
        else half_tile<TWO, STRONG>(xr + A::GY, xr + A::V, out, tx, ty, t4, l16, g);
    };
    F4 c2e = {}, c2m = {}, c2k = {};
    float u2 = 0.f, w24 = 1.f, gw2 = 0.f, gu2 = 0.f;
    const float l2 = S.hd.lam2[own];
    if constexpr (TWO) {
        u2 = S.hd.u2[own]; w24 = wpow(l2, 4.f);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 4 * g + v, m = ref<STRONG>(t);
            c2e[v] = wpow(l2, static_cast<float>(15 - t));
            c2m[v] = wpow(l2, static_cast<float>(t - m)); c2k[v] = wpow(l2, static_cast<float>(m - 1 - t));
            lag[v] = static_cast<float>(l16 - 1 - t);
        }
    }
    __syncthreads();
    tile(nch - 1);
    __syncthreads();
    auto chunk = [&](const int c) __attribute__((always_inline)) {
        const uint32_t sx = A::slot(c), xr = hide(sx + orow), xc = hide(sx + ocol), xg = hide(sx + 16 * g);
        const uint32_t dt0 = hide(A::ds(c) + odt), tc = hide(A::tile(c, 0) + otc);
        f32x4 go, aT;
        f32x4 y2[2] = {ZERO4, ZERO4};
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
            const f32x4 ka = lds4(xr + A::K + 64 * jt) * cke[jt], dt = lds4(dt0 + 64 * jt);
#pragma unroll
            for (int v = 0; v < 4; ++v) y2[jt & 1] = mm(ka[v], dt[v], y2[jt & 1]);
        }
        go = col4(xc + A::GY); aT = col4<TROWB>(tc) + col4<TROWB>(tc + TILEB);
        const f32x4 ruk = lds4(xg + A::RUK);
        f32x4 dv = y2[0] + y2[1];
        if constexpr (TWO) {
            const f32x4 rk = lds4(xg + A::RK), gm = go * c2m, vo = col4(xc + A::V);
            dv = dv * c2e + apply<STRONG>(aT, gm, l16 < 8 && g >= 2, w24) * c2k + go * (ruk + u2 * rk);
            const uint32_t tr = hide(A::tile(c, 0) + otr);
            const f32x4 a = lds4(tr) + lds4(tr + TILEB);
            gw2 += sum4(gm * apply<STRONG>(a * lag, vo * c2k, l16 >= 8 && g < 2, w24));
            gu2 += sum4(vo * go * rk);
        } else {
            dv += go * ruk;
#pragma unroll
            for (int v = 0; v < 4; ++v) dv = mm(aT[v], go[v], dv);
        }
        store_chunk(p.gv, base, c, g, own, C, T, dv);
        if (c > 0) tile(c - 1);
    };
    for (int s = (nch - 1) / G; s >= 0; --s) {
#pragma unroll
        for (int z = G - 1; z >= 0; --z) {
            const int c = s * G + z;
            if (c < nch) {
                chunk(c);
                if (c >= G) put(c - G, ring[z]);
                fetch(c - 2 * G, ring[z]);
                __syncthreads();
            }
        }
    }
    __syncthreads();
    if (q == 0 && lane == 0 && S.marked && p.NB == 1) mark(p.gv + base);
    if constexpr (TWO) {
        gw2 = allreduce_rows(gw2); gu2 = allreduce_rows(gu2);
        if (g == 0) {
            const size_t o = (static_cast<size_t>(part.n) * p.B + part.b) * C + part.h * N + own;
#pragma unroll
            for (int z = 0; z < 4; ++z) gw2 += S.red[z][own];
            p.gw2[o] = l2 * gw2;
            p.gu2[o] = gu2;
        }
    }
}

template <bool TWO, bool STRONG>
DEVINL void bwd_roles(SmemB<TWO>& S, const ArgsC& p, int w, int lane, const Part<TWO>& part) {
    const int q = w & 3;
    if (w < 4) role_d<TWO, STRONG>(S, p, q, lane, part);
    else role_e<TWO, STRONG>(S, p, q, lane, part);
}

template <bool TWO, bool CUT>
__global__ __launch_bounds__(NTB, 2) void wkv5c_bwd(const ArgsC args) {
    const ArgsC p = only_whole<CUT>(args);
    SmemB<TWO>& S = *reinterpret_cast<SmemB<TWO>*>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Part<TWO> part = part_of<TWO>(p);
    if (steps_head<true, N>(p.w, TWO ? p.w2 : nullptr, part.h * N)) return;
    const bool strong = head_setup<TWO>(S.hd, p, part.h, tid);
    if (tid == 0) S.marked = 0;
    __syncthreads();
    if (strong) bwd_roles<TWO, true>(S, p, w, lane, part);
    else bwd_roles<TWO, false>(S, p, w, lane, part);
}

// out[c] = sum over blocks and batch of the rows of up to four [NB][B][C] arrays that lie behind each other.  A head that the step kernels
// have done has its sum in the first of its blocks' rows.
__global__ __launch_bounds__(256) void rows_sum(int B, int C, int NB, const int* __restrict__ flags, const float* __restrict__ rows, float* o0, float* o1, float* o2, float* o3) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const float* x = rows + static_cast<size_t>(blockIdx.y) * NB * B * C + c;
    float s = 0.f;
    for (int b = 0; b < B; ++b) {
        const int blocks = NB > 1 && flags[b * (C / N) + c / N] == 0 ? NB : 1;
        float t = 0.f;
        for (int n = 0; n < blocks; ++n) t += x[(static_cast<size_t>(n) * B + b) * C];
        s += t;
    }
    (blockIdx.y == 0 ? o0 : (blockIdx.y == 1 ? o1 : (blockIdx.y == 2 ? o2 : o3)))[c] = s;
}

// Blocks of time: as many as there is room for on the card at a time (two workgroups a CU in the forward, one in the backward), of
// BLOCK_SEGS segments at least; 1: whole sequences.  per: segments a block.  Where the line lies, B H sequences, us as they are whole / in
// blocks: wkv5 forward 8 of T400 41 / 26, of T4096 355 / 62; 64 of T400 42 / 36, of T4096 360 / 146; 128 of T400 43 / 45, of T800 76 / 75, of
// T4096 358 / 246; 192 (two blocks) of T800 78 / 85, of T4096 360 / 349.  Forward + backward of T4096: 8 sequences 1015 / 129, 32
// 1022 / 232, 128 1056 / 691; wkv5a 1252 / 160, 1276 / 267, 1301 / 789.  Below some 300 tokens the launch in front takes what the blocks save.
constexpr int BLOCK_SEGS = 2, SLOTS_FWD = 512, SLOTS_BWD = 256;
template <bool TWO> int time_blocks(int B, int T, int H, bool bwd, int* per) {
    const long long bh = static_cast<long long>(B) * H;
    const int nch = static_cast<int>((static_cast<long long>(T) + L - 1) / L), nseg = (nch + SEG<TWO> - 1) / SEG<TWO>;
    *per = nseg;
    const long long want = (bwd ? SLOTS_BWD : SLOTS_FWD) / bh;
    if (want < (bwd ? 2 : 4) || nch < 16 + bh / 4) return 1;
    const int least = static_cast<int>((nseg + want - 1) / want);
    *per = least > BLOCK_SEGS ? least : BLOCK_SEGS;
    return (nseg + *per - 1) / *per;
}
// bytes of the blocks' states and of the heads' words
size_t blocks_bytes(int B, int H, int NB) {
    const size_t bh = static_cast<size_t>(B) * H;
    return NB > 1 ? bh * (NB - 1) * N * N * sizeof(float) + (bh * sizeof(int) + 15) / 16 * 16 : 0;
}
template <bool TWO> void set_blocks(ArgsC& p, int B, int NB, int per, void* ws) {
    p.B = B; p.NB = NB; p.per = per;
    if (NB > 1) {
        p.local = static_cast<float*>(ws);
        p.flags = reinterpret_cast<int*>(p.local + static_cast<size_t>(B) * p.H * (NB - 1) * N * N);
    }
}

template <bool TWO> size_t saved_bytes(int B, int T, int C, int H) {
    if (B <= 0 || T <= 0 || H <= 0 || C != H * N) return 0;
    const size_t nch = (static_cast<size_t>(T) + L - 1) / L;
    return static_cast<size_t>(B) * H * ((nch + SEG<TWO> - 1) / SEG<TWO>) * N * N * sizeof(float);
}
int check(int B, int T, int C, int H) {
    if (B <= 0 || T <= 0 || H <= 0 || C != H * N) return RWKV_ERR_SHAPE;
    if (static_cast<long long>(B) * H > 0x7fffffffLL || C > (1 << 26)) return RWKV_ERR_SHAPE;      // 16 rows by a 32-bit offset
    return RWKV_OK;
}

template <bool TWO> size_t fwd_ws_bytes(int B, int T, int C, int H) {
    int per;
    return check(B, T, C, H) == RWKV_OK ? blocks_bytes(B, H, time_blocks<TWO>(B, T, H, false, &per)) : 0;
}
// per-block and per-batch rows of the parameters' gradients, then what the blocks take
template <bool TWO> size_t bwd_rows_bytes(int B, int C, int NB) { return ((TWO ? 4 : 2) * static_cast<size_t>(NB) * B * C * sizeof(float) + 15) / 16 * 16; }
template <bool TWO> size_t bwd_ws_bytes(int B, int T, int C, int H) {
    if (check(B, T, C, H) != RWKV_OK) return 0;
    int per;
    const int NB = time_blocks<TWO>(B, T, H, true, &per);
    return bwd_rows_bytes<TWO>(B, C, NB) + blocks_bytes(B, H, NB);
}
template <bool TWO> int start_fwd(void* stream, int B, ArgsC& p, void* ws, size_t ws_bytes) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    int per = 0, NB = 1;
    if (ws != nullptr) {
        if (ws_bytes < fwd_ws_bytes<TWO>(B, p.T, p.C, p.H) || !aligned16(ws)) return RWKV_ERR_WORKSPACE;
        NB = time_blocks<TWO>(B, p.T, p.H, false, &per);
    }
    set_blocks<TWO>(p, B, NB, per, ws);
    if (NB > 1) hipLaunchKernelGGL((wkv5c_local<TWO, false>), dim3(B * p.H * (NB - 1) * 4), dim3(256), 0, st, p);
    hipLaunchKernelGGL((NB > 1 ? wkv5c_fwd<TWO, true> : wkv5c_fwd<TWO, false>), dim3(B * p.H * NB), dim3(NT), 0, st, p);
    return launch_wkv5f32_steps_fwd(st, B, p.T, p.H, p.r, p.k, p.v, p.w, p.u, p.w2, p.u2, p.y, p.flags);
}
hipError_t raise_lds(void (*kernel)(ArgsC), size_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
}
// (a workspace that holds the rows of whole sequences and no more, or that the blocks' 16-byte accesses do not fit, is for whole sequences: they
// take single floats)
template <bool TWO> int start_bwd(void* stream, int B, ArgsC& p, void* ws, size_t ws_bytes, float* gw, float* gu, float* gw2, float* gu2) {
    if (ws == nullptr || ws_bytes < bwd_rows_bytes<TWO>(B, p.C, 1)) return RWKV_ERR_WORKSPACE;
    static_assert(sizeof(SmemB<TWO>) <= 160 * 1024, "the backward's LDS must fit one CU");
    static const hipError_t attr[2] = {raise_lds(wkv5c_bwd<TWO, false>, sizeof(SmemB<TWO>)), raise_lds(wkv5c_bwd<TWO, true>, sizeof(SmemB<TWO>))};
    for (const hipError_t e : attr) if (e != hipSuccess) { g_last_hip_error = static_cast<int>(e); return RWKV_ERR_LAUNCH; }
    hipStream_t st = static_cast<hipStream_t>(stream);
    int per = 0;
    const int NB = ws_bytes < bwd_ws_bytes<TWO>(B, p.T, p.C, p.H) || !aligned16(ws) ? 1 : time_blocks<TWO>(B, p.T, p.H, true, &per);
    const size_t m = static_cast<size_t>(NB) * B * p.C;
    float* const rows = static_cast<float*>(ws);
    p.gw = rows; p.gu = rows + m;
    if constexpr (TWO) { p.gw2 = rows + 2 * m; p.gu2 = rows + 3 * m; }
    set_blocks<TWO>(p, B, NB, per, static_cast<char*>(ws) + bwd_rows_bytes<TWO>(B, p.C, NB));
    if (NB > 1) hipLaunchKernelGGL((wkv5c_local<TWO, true>), dim3(B * p.H * (NB - 1) * 4), dim3(256), 0, st, p);
    hipLaunchKernelGGL((NB > 1 ? wkv5c_bwd<TWO, true> : wkv5c_bwd<TWO, false>), dim3(B * p.H * NB), dim3(NTB), sizeof(SmemB<TWO>), st, p);
    if (int e = launch_wkv5f32_steps_bwd(st, B, p.T, p.H, p.r, p.k, p.v, p.w, p.u, p.w2, p.u2, p.gy, p.gr, p.gk, p.gv, p.gw, p.gu, p.gw2, p.gu2, p.flags)) return e;
    hipLaunchKernelGGL(rows_sum, dim3((p.C + 255) / 256, TWO ? 4 : 2), dim3(256), 0, st, B, p.C, NB, p.flags, rows, gw, gu, gw2, gu2);
    return launch_status();
}

}  // namespace
}  // namespace rwkv

using namespace rwkv;

extern "C" {

size_t rwkv_wkv5f32s_saved_bytes(int B, int T, int C, int H) { return saved_bytes<false>(B, T, C, H); }
size_t rwkv_wkv5as_saved_bytes(int B, int T, int C, int H) { return saved_bytes<true>(B, T, C, H); }
size_t rwkv_wkv5f32s_forward_workspace_bytes(int B, int T, int C, int H) { return fwd_ws_bytes<false>(B, T, C, H); }
size_t rwkv_wkv5as_forward_workspace_bytes(int B, int T, int C, int H) { return fwd_ws_bytes<true>(B, T, C, H); }
size_t rwkv_wkv5f32s_backward_workspace_bytes(int B, int T, int C, int H) { return bwd_ws_bytes<false>(B, T, C, H); }
size_t rwkv_wkv5as_backward_workspace_bytes(int B, int T, int C, int H) { return bwd_ws_bytes<true>(B, T, C, H); }

int rwkv_wkv5f32s_forward_ws(void* stream, int B, int T, int C, int H, const float* r, const float* k, const float* v, const float* w,
                             const float* u, float* y, void* saved, size_t bytes, void* workspace, size_t workspace_bytes) {
    if (int e = check(B, T, C, H)) return e;
    if (int e = check_ptrs({r, k, v, u, y})) return e;
    if (int e = check_ptrs({w}, false)) return e;
    if (saved != nullptr && (bytes < saved_bytes<false>(B, T, C, H) || !aligned16(saved))) return RWKV_ERR_WORKSPACE;
    ArgsC p{};
    p.T = T; p.C = C; p.H = H; p.r = r; p.k = k; p.v = v; p.w = w; p.u = u; p.y = y; p.saved = static_cast<float*>(saved);
    return start_fwd<false>(stream, B, p, workspace, workspace_bytes);
}
int rwkv_wkv5f32s_forward(void* stream, int B, int T, int C, int H, const float* r, const float* k, const float* v, const float* w,
                          const float* u, float* y, void* saved, size_t bytes) {
    return rwkv_wkv5f32s_forward_ws(stream, B, T, C, H, r, k, v, w, u, y, saved, bytes, nullptr, 0);
}

int rwkv_wkv5f32s_backward(void* stream, int B, int T, int C, int H, const float* r, const float* k, const float* v, const float* w,
                           const float* u, const float* gy, float* gr, float* gk, float* gv, float* gw, float* gu, const void* saved,
                           size_t bytes, void* workspace, size_t workspace_bytes) {
    if (int e = check(B, T, C, H)) return e;
    if (int e = check_ptrs({r, k, v, u, gy, gr, gk, gv, gw, gu})) return e;
    if (int e = check_ptrs({w}, false)) return e;
    if (saved == nullptr || bytes < saved_bytes<false>(B, T, C, H) || !aligned16(saved)) return RWKV_ERR_WORKSPACE;
    ArgsC p{};
    p.T = T; p.C = C; p.H = H; p.r = r; p.k = k; p.v = v; p.w = w; p.u = u; p.gy = gy; p.gr = gr; p.gk = gk; p.gv = gv;
    p.saved = static_cast<float*>(const_cast<void*>(saved));
    return start_bwd<false>(stream, B, p, workspace, workspace_bytes, gw, gu, nullptr, nullptr);
}

int rwkv_wkv5as_forward_ws(void* stream, int B, int T, int C, int H, const float* r, const float* k, const float* v, const float* w1,
                           const float* u1, const float* w2, const float* u2, float* y, void* saved, size_t bytes, void* workspace,
                           size_t workspace_bytes) {
    if (int e = check(B, T, C, H)) return e;
    if (int e = check_ptrs({r, k, v, u1, u2, y})) return e;
    if (int e = check_ptrs({w1, w2}, false)) return e;
    if (saved != nullptr && (bytes < saved_bytes<true>(B, T, C, H) || !aligned16(saved))) return RWKV_ERR_WORKSPACE;
    ArgsC p{};
    p.T = T; p.C = C; p.H = H; p.r = r; p.k = k; p.v = v; p.w = w1; p.u = u1; p.w2 = w2; p.u2 = u2; p.y = y;
    p.saved = static_cast<float*>(saved);
    return start_fwd<true>(stream, B, p, workspace, workspace_bytes);
}
int rwkv_wkv5as_forward(void* stream, int B, int T, int C, int H, const float* r, const float* k, const float* v, const float* w1,
                        const float* u1, const float* w2, const float* u2, float* y, void* saved, size_t bytes) {
    return rwkv_wkv5as_forward_ws(stream, B, T, C, H, r, k, v, w1, u1, w2, u2, y, saved, bytes, nullptr, 0);
}

int rwkv_wkv5as_backward(void* stream, int B, int T, int C, int H, const float* r, const float* k, const float* v, const float* w1,
                         const float* u1, const float* w2, const float* u2, const float* gy, float* gr, float* gk, float* gv,
                         float* gw1, float* gu1, float* gw2, float* gu2, const void* saved, size_t bytes, void* workspace,
                         size_t workspace_bytes) {
    if (int e = check(B, T, C, H)) return e;
    if (int e = check_ptrs({r, k, v, u1, u2, gy, gr, gk, gv, gw1, gu1, gw2, gu2})) return e;
    if (int e = check_ptrs({w1, w2}, false)) return e;
    if (saved == nullptr || bytes < saved_bytes<true>(B, T, C, H) || !aligned16(saved)) return RWKV_ERR_WORKSPACE;
    ArgsC p{};
    p.T = T; p.C = C; p.H = H; p.r = r; p.k = k; p.v = v; p.w = w1; p.u = u1; p.w2 = w2; p.u2 = u2; p.gy = gy;
    p.gr = gr; p.gk = gk; p.gv = gv; p.saved = static_cast<float*>(const_cast<void*>(saved));
    return start_bwd<true>(stream, B, p, workspace, workspace_bytes, gw1, gu1, gw2, gu2);
}

}  // extern "C"
