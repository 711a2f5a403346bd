// wkv5, bf16 I/O, whole heads of N = 128 or 64 channels in one workgroup: one forward and one reverse sweep in chunks of
// L = 32 tokens on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16), for decays up to e^-9 a step.
//
// Step form (wkv5_bf16/cuda/wkv5_cuda.cu), one head, S[i][j] (i value channel, j key channel), o = e^l, l = -exp(w_raw):
//     y_t[i] = sum_j r_t[j] (S_t[i][j] + u[j] k_t[j] v_t[i])       S_{t+1} = S_t o + v_t k_t^T
// The decay is constant in time, so the powers a token of a chunk (local t = 0..31) needs are the same in every chunk and are
// made once per workgroup.  S0 is the state entering the chunk, D the gradient of the state leaving it, m a reference token:
//     A[t][s] = sum_j (r_t o^{t-m}) (k_s o^{m-1-s})  (s < t), A[t][t] = sum_j r_t u k_t        B[t][s] = gy_t . v_s  (s < t)
//     y_t  = (r_t o^t) S0^T + sum_s A[t][s] v_s
//     gr_t = o^t (gy_t S0) + o^{t-m} sum_s B[t][s] (k_s o^{m-1-s}) + u k_t (v_t . gy_t)
//     gk_t = o^{31-t} (v_t D) + o^{m-1-t} sum_s B[s][t] (r_s o^{s-m}) + u r_t (v_t . gy_t)
//     gv_t = (k_t o^{31-t}) D^T + sum_s A[s][t] gy_s
//     S_L = S0 o^32 + sum_s v_s (k_s o^{31-s})^T           D_0 = D o^32 + sum_t gy_t (r_t o^t)^T
// A term (source s, sink t) of the output carries o^(tokens strictly between), so d/dl counts those tokens: t for sources before
// the chunk, 31 - s for sinks after it, 32 where both lie outside, t - 1 - s inside (the tile B with this weight; taken apart into
// (t - 16) - (s - 15) the sums would cancel, and two hi / lo products differ by 1e-5 where the true gradient is zero).
// Operands: fp32 values as hi + lo bf16 (16 mantissa bits), three products where both sides are fp32; r, k, v, gy are exact.
//
// Strong decays.  A factor reaches e^{|l| d}, d the distance of a token from its reference.  The forward has one reference in the
// middle (its planes serve the state products too), up to |l| = 4.5, and makes its tiles from raw rows beyond.  These, and the
// backward always, refer to the middle of the half that the output's token lies in (m = 8, 24; a tile's quadrant across the halves
// to 16): d is 8 and |l| may reach 9, for one more operand per tile.  A head beyond that, or with a decay that is no number, is left
// to wkv5_steps_* (steps_head, common.h): with a reference per 8 tokens, and a product for each distance of two such blocks, the
// loops spill hundreds of registers, and decays below e^-17 are out of reach all the same.
// Handing every head with a strong decay (|l| > 3.7) to step-by-step kernels, as the kernels before did, made one such channel in
// 4096 cost more than everything else: B8 T4096 C4096 N128, forward + backward, 3.8 ms without one, 6.6 to 11.3 ms with.  That is
// why layers of 64-channel heads come here as well once they have such a channel (B8 T4096 C2048: 0.69 ms with a channel at
// l = -4.5 or -8.6, where they took 1.7 to 3.8 ms).
//
// What bounds it (B8 T4096 C4096: one workgroup per CU).  Forward 0.43 ms for 2.1 GB, half of them the saved states: HBM (5.0 TB/s;
// 0.82 ms as four heads of 64).  Backward 0.98 ms, 3.3 GB: memory and issue, which its two barriers a chunk do not let overlap
// entirely (2.95 ms as two sweeps over four heads of 64, whose fp32 terms went through memory).  Both together 6.56 -> 1.48 ms where a
// channel's decay was strong, 3.83 -> 1.43 where none was.
#include <stddef.h>

#include "wkv6_fused.h"

namespace rwkv {
namespace {

constexpr int NTH = 512;             // forward: waves 0..3 hold states, 4..7 load and prepare
constexpr float LAM_MID = -4.5f;     // strongest log decay for one reference (one per half: W_STEPS_BF16)
constexpr f32x4 ZERO4 = {0.f, 0.f, 0.f, 0.f};

struct ArgsW {
    int T, C, H;
    const uint16_t *r, *k, *v, *w, *u, *gy;      // w raw
    uint16_t *y, *gr, *gk, *gv, *gw, *gu;        // gw, gu: per-batch rows [B][C]
    float* decay;                                // [e^l | l], 2 C floats (forward)
    float* saved;                                // [B*H][ceil(chunks / 2)][j][i]: the state entering every even chunk
    // sequences cut into blocks of time (NB > 1): blocks of `per` pairs of chunks, a workgroup each; what each block leaves of a state that
    // entered it empty, [heads][NB - 1][HN][HN] (the last block's is not needed, in the backward the first's); gw, gu in fp32 [NB][heads][HN].
    // heads: of this launch, from head `at` on, batch row by batch row
    int heads, at, NB, per;
    float *local, *gw32, *gu32;
};

// The workgroup's head and its part of the sequence: chunks first .. first + chunks - 1, tokens that are left from there on.
struct Part {
    int h, b, rel, n, first, chunks, left;      // rel: among the launch's heads
    size_t bh, base;
};
// pairs: an odd number of chunks is rounded up
DEVINL Part part_of(const ArgsW& p, int hn, bool pairs) {
    Part x;
    int nch = (p.T + L - 1) / L;
    if (pairs) nch += nch & 1;
    // (divisions are done in vector registers)
    x.n = __builtin_amdgcn_readfirstlane(p.NB > 1 ? static_cast<int>(blockIdx.x) / p.heads : 0);
    x.rel = blockIdx.x - x.n * p.heads;
    x.bh = p.at + x.rel;
    x.b = __builtin_amdgcn_readfirstlane(static_cast<int>(x.bh) / p.H); x.h = static_cast<int>(x.bh) - x.b * p.H;
    x.first = x.n * 2 * p.per;
    x.chunks = p.NB > 1 ? min(2 * p.per, nch - x.first) : nch;
    x.left = p.T - x.first * L;
    x.base = (static_cast<size_t>(x.b) * p.T + static_cast<size_t>(x.first) * L) * p.C + static_cast<size_t>(x.h) * hn;
    return x;
}
// where the states of the part's pairs of chunks are
template <int HN> DEVINL float* saved_state(const ArgsW& p, const Part& x) {
    return p.saved + (x.bh * ((p.T + 2 * L - 1) / (2 * L)) + x.first / 2) * HN * HN;
}

extern __shared__ __align__(16) unsigned char smem_raw[];

// Sizes of one head.  A wave owns CT tiles of 16 channels; a row of 2 N bytes is loaded in PIECES of 16 bytes.
template <int HN> struct G {
    static constexpr int CT = HN / 64, KS = HN / 32, NB16 = HN / 16, PARTS = HN / 32;
    static constexpr int PIECES = HN / 8, ROWS = 256 / PIECES, PASSES = L / ROWS;
    static constexpr uint32_t ROW = 2 * HN + 16, PLANE = L * ROW;
    static constexpr uint32_t LAM = 0, U = 4 * HN, BLK = 8 * HN, BASE = 12 * HN;      // BLK: decay of a block of time
    static constexpr uint32_t PART = 3 * 1024;                                   // the three quadrants of a tile, fp32, as the lanes hold them
    // forward: three slots of planes R' hi, lo, K' hi, lo, V and sum r u k; two sets of tile parts
    static constexpr uint32_t FRH = 0, FRL = PLANE, FKH = 2 * PLANE, FKL = 3 * PLANE, FV = 4 * PLANE, FRUK = 5 * PLANE, FSLOT = FRUK + 4 * L;
    static constexpr uint32_t FPART = BASE + 3 * FSLOT, FTOTAL = FPART + 2 * PARTS * PART;
    // backward: two slots of planes r, k, v, gy and two scalars a token; the gradient state hi, lo [j][i]; one set of parts of tile A; tile B in three forms
    static constexpr uint32_t R = 0, K = PLANE, V = 2 * PLANE, GY = 3 * PLANE, VG = 4 * PLANE, RUK = VG + 4 * L, SLOT = RUK + 4 * L;
    static constexpr uint32_t DSH = BASE + 2 * SLOT, DSL = DSH + HN * ROW, BPART = DSL + HN * ROW, BTILE = BPART + PARTS * PART, BTOTAL = BTILE + 3 * PART;
};
static_assert(G<128>::FTOTAL <= 160 * 1024 && G<128>::BTOTAL <= 160 * 1024, "LDS of one CU");

DEVINL float lds_f(uint32_t o) { return lds_ld<float>(o); }

// e^{lam n} for a small integer n, exact to fp32 rounding: the product and the base-2 exponent carry their rounding errors along
DEVINL float wpow(float lam, float n) {
    constexpr float L2E_HI = 1.44269502162933349609f, L2E_LO = 1.92596299112661746e-8f, LN2F = 0.69314718055994530942f;
    const float x = lam * n, lo = fmaf(lam, n, -x);
    const float t = x * L2E_HI;
    const float e = fmaf(x, L2E_HI, -t) + fmaf(x, L2E_LO, lo * L2E_HI);
    const float y = __builtin_amdgcn_exp2f(t);
    float r = fmaf(y, e * LN2F, y);
    asm volatile("" : "+v"(r));
    return r;
}
DEVINL float wpow(float lam, int n) { return wpow(lam, static_cast<float>(n)); }

template <int CTRL> DEVINL float dpp(float x) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true)); }
// sum over groups of 8 or 16 lanes, in all of them
template <int LANES> DEVINL float lanes_sum(float x) {
    x += dpp<0xB1>(x); x += dpp<0x4E>(x); x += dpp<0x141>(x);      // lane ^ 1, lane ^ 2, mirrored within eight
    if constexpr (LANES == 16) x += dpp<0x140>(x);                // mirrored within sixteen
    return x;
}
// eight fp32 values -> hi and lo operands
struct Op2 { bf16x8 h, l; };
DEVINL Op2 split8(const float (&x)[8]) {
    const HL a = hilo2k(x[0], x[1]), b = hilo2k(x[2], x[3]), c = hilo2k(x[4], x[5]), d = hilo2k(x[6], x[7]);
    return {as_op(a.h, b.h, c.h, d.h), as_op(a.l, b.l, c.l, d.l)};
}
DEVINL Op2 split8(const f32x4& x, const f32x4& y) { const float f[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}; return split8(f); }
DEVINL f32x4 mm3(const Op2& a, const Op2& b, f32x4 c) { return mfma(a.l, b.h, mfma(a.h, b.l, mfma(a.h, b.h, c))); }
DEVINL void unpack(const bf16x8& x, float (&f)[8]) { unpack8(__builtin_bit_cast(uint4, x), f); }
// hi and lo of the products a p and b q; the remainders are those of the exact products.  (Written as a product and its split, they are that
// where the compiler finds both in one basic block, and of the rounded product elsewhere.)
DEVINL HL hilo2p(float a, float p, float b, float q) {
    HL r;
    r.h = cvt2(a * p, b * q);
    asm("" : "+v"(r.h));
    r.l = cvt2(fmaf(a, p, -__uint_as_float(r.h << 16)), fmaf(b, q, -__uint_as_float(r.h & 0xffff0000u)));
    return r;
}
DEVINL Op2 scaled(const bf16x8& x, const float (&p)[8]) {
    float f[8];
    unpack(x, f);
    const HL a = hilo2p(f[0], p[0], f[1], p[1]), b = hilo2p(f[2], p[2], f[3], p[3]), c = hilo2p(f[4], p[4], f[5], p[5]), d = hilo2p(f[6], p[6], f[7], p[7]);
    return {as_op(a.h, b.h, c.h, d.h), as_op(a.l, b.l, c.l, d.l)};
}
// Operand with the 32 rows (tokens) of a plane along K in accumulator order: slot (g, e) <-> row 16 (e >> 2) + 4 g + (e & 3), lane
// <-> column.  a: element [4 g + (l16 >> 2)][col + 4 (l16 & 3)].
template <uint32_t ROW> DEVINL bf16x8 ld_tra(const lds_t a) {
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(a));
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(a + 16 * ROW));
    const u32x2 x = __builtin_bit_cast(u32x2, lo), y = __builtin_bit_cast(u32x2, hi);
    return as_op(x[0], x[1], y[0], y[1]);
}
DEVINL int slot_token(int g, int e) { return 16 * (e >> 2) + 4 * g + (e & 3); }

// The head's parameters into LDS (by the first wave); every wave finds out for itself what its strongest log decay is.
template <int HN> DEVINL float head_setup(const ArgsW& p, lds_t sb, const Part& part, int tid) {
    const int lane = tid & 63;
    float mn = 0.f;
#pragma unroll
    for (int z = 0; z < HN / 64; ++z) {
        const int n = 64 * z + lane, c = part.h * HN + n;
        const float l = -expf(bf2f(p.w[c]));
        mn = fminf(mn, l);
        if (tid < 64) {
            lds_st<float>(sb + G<HN>::LAM + 4 * n, l);
            lds_st<float>(sb + G<HN>::U + 4 * n, bf2f(p.u[c]));
            lds_st<float>(sb + G<HN>::BLK + 4 * n, wpow(l, 2 * L * p.per));
            if (p.decay != nullptr && part.b == 0 && part.n == 0) { p.decay[c] = expf(l); p.decay[p.C + c] = l; }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o, 64));
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, mn)));
}

// Rows of a [token][channel] tensor from one token on, as a buffer: reads of rows that do not exist give zeros, stores to them are
// dropped, so the ends of a sequence cost no branches and no masks (an offset of 32 rows stays below 2^31: WKV5B_MAX_C).
typedef __amdgpu_buffer_rsrc_t rows_t;
DEVINL rows_t rows_of(const uint16_t* first, int left, int C) {
    // (the two limits become one vector instruction: its result has to come back for the descriptor)
    const int rows = __builtin_amdgcn_readfirstlane(min(max(left, 0), L));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(first), 0, rows * C * 2, 0x00027000);
}
DEVINL uint4 load16(rows_t r, int o) { return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0)); }

// A 16 x 16 tile of a bf16 output: rows (tokens) 4 g + v, lane = column.  Neighbouring lanes exchange halves, so that each stores
// pairs of columns: even lanes rows 4 g, 4 g + 1, odd lanes the other two.  o: byte offset of the lane's first row and column.
DEVINL int tile_offset(int l16, int g, int C) { return (4 * g + 2 * (l16 & 1)) * 2 * C + 2 * (l16 & ~1); }
DEVINL void store_tile(rows_t out, int o, int C, int l16, const f32x4& x) {
    const bool odd = l16 & 1;
    const float r0 = dpp<0xB1>(odd ? x[0] : x[2]), r1 = dpp<0xB1>(odd ? x[1] : x[3]);
    const uint32_t a = cvt2(odd ? r0 : x[0], odd ? x[2] : r0), b = cvt2(odd ? r1 : x[1], odd ? x[3] : r1);
    __builtin_amdgcn_raw_buffer_store_b32(a, out, o, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32(b, out, o + 2 * C, 0, 0);
}

// One wave's part (32 channels of the contraction) of a causal tile D[snk][src] = sum_j x_snk y_src, src <= snk, lane = src or snk
// (LANE_SNK): three quadrants (row tile, lane tile).  x, y: two operands each (token tiles).
template <bool LANE_SNK> struct Quad {       // {row tile, lane tile} of quadrant z
    static constexpr int ROWT[3] = {0, LANE_SNK ? 0 : 1, 1}, LANET[3] = {0, LANE_SNK ? 1 : 0, 1};
};
// lane and row token of a tile element, whether it is strictly causal
template <bool LANE_SNK> DEVINL bool causal(int z, int l16, int row) {
    const int a = 16 * Quad<LANE_SNK>::ROWT[z] + row, b = 16 * Quad<LANE_SNK>::LANET[z] + l16;
    return LANE_SNK ? a < b : b < a;
}
// a quadrant of the part, masked, with `diag` (of the lane's token) on its diagonal, to LDS
template <bool LANE_SNK, int z> DEVINL void put_quad(lds_t out, const f32x4& q, float diag, int lane) {
    const int l16 = lane & 15, g = lane >> 4;
    f32x4 x;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        x[v] = causal<LANE_SNK>(z, l16, 4 * g + v) ? q[v] : 0.f;
        if (Quad<LANE_SNK>::ROWT[z] == Quad<LANE_SNK>::LANET[z]) x[v] = l16 == 4 * g + v ? diag : x[v];
    }
    lds_st<f32x4>(out + 1024 * z + 16 * lane, x);
}
// the parts added up and split: operands of the two lane tiles (slots: the row tokens in accumulator order)
template <int PARTS, uint32_t PART> DEVINL f32x4 sum_parts(lds_t in, int z, int lane) {
    f32x4 s = lds_ld<f32x4>(in + 1024 * z + 16 * lane);
#pragma unroll
    for (int i = 1; i < PARTS; ++i) s += lds_ld<f32x4>(in + i * PART + 1024 * z + 16 * lane);
    return s;
}
// lane is the sink (forward): sources of tile 0 for both lane tiles, of tile 1 for the second
template <int PARTS, uint32_t PART> DEVINL void take_parts(lds_t in, int lane, Op2 (&a)[2]) {
    a[0] = split8(sum_parts<PARTS, PART>(in, 0, lane), ZERO4);
    a[1] = split8(sum_parts<PARTS, PART>(in, 1, lane), sum_parts<PARTS, PART>(in, 2, lane));
}
// lane is the source (backward): the other way round; one lane tile
template <int PARTS, uint32_t PART, int Z> DEVINL Op2 take_lane_tile(lds_t in, int lane) {
    if constexpr (Z == 0) return split8(sum_parts<PARTS, PART>(in, 0, lane), sum_parts<PARTS, PART>(in, 1, lane));
    else return split8(ZERO4, sum_parts<PARTS, PART>(in, 2, lane));
}
// powers for a tile part, channel ch0 + e: of token 16 z + l16, x as the sink, y as the source; they are those of the token in its
// half and serve both.  cx, cy: as sink of the second and source of the first half of a pair across them.
struct TilePowers { float px[8], py[8], cx[8], cy[8]; };
DEVINL void tile_powers(TilePowers& t, lds_t lam, int l16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float l = lds_f(lam + 4 * e);
        t.px[e] = wpow(l, l16 - 8); t.py[e] = wpow(l, 7 - l16);
        t.cx[e] = wpow(l, l16); t.cy[e] = wpow(l, 15 - l16);
    }
}
// tile part from raw rows (operands of the two token tiles), lane = sink
DEVINL void raw_part(const bf16x8 (&r)[2], const bf16x8 (&k)[2], const TilePowers& t, f32x4 (&q)[3]) {
    using Q = Quad<true>;
#pragma unroll
    for (int z = 0; z < 3; ++z) {
        const bool across = Q::ROWT[z] != Q::LANET[z];
        const Op2 x = scaled(r[Q::LANET[z]], across ? t.cx : t.px), y = scaled(k[Q::ROWT[z]], across ? t.cy : t.py);
        q[z] = mm3(y, x, ZERO4);
    }
}

// ---------------------------------------------------------------------------------------------------- blocks of time, first pass
// What a block leaves of an empty state: sum over its tokens of v_t k_t^T with the decay that is left to the block's end, stored as [i][j]
// for the forward, or (REV) from the end backwards what the gradient state takes up, gy_t r_t^T, stored as [j][i] for the D waves.  A wave
// makes 32 key channels, whose operand takes the powers (hi + lo); the other side is exact.
template <int HN, bool REV>
__global__ __launch_bounds__(256) void wkv5b_local(const ArgsW p) {
    using A = G<HN>;
    constexpr int NT = A::NB16, NP = A::PASSES, CT = A::CT;
    __shared__ __align__(16) unsigned char rows[4 * A::PLANE];           // two sets of key and value rows
    const lds_t sb = lds_of(rows);
    const int tid = threadIdx.x, lane = tid & 63, q = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4, C = p.C;
    const int m = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) / p.heads), rel = blockIdx.x - m * p.heads, bh = p.at + rel;
    const int b = __builtin_amdgcn_readfirstlane(bh / p.H), h = bh - b * p.H, n = REV ? m + 1 : m;
    if (steps_head<false, HN>(p.w, nullptr, h * HN)) return;
    const int first = n * 2 * p.per, chunks = min(2 * p.per, (p.T + L - 1) / L - first);
    const size_t base = (static_cast<size_t>(b) * p.T + static_cast<size_t>(first) * L) * C + static_cast<size_t>(h) * HN;
    const int left = p.T - first * L, row0 = tid / A::PIECES, c8 = (tid % A::PIECES) * 8;
    const uint16_t* const key = (REV ? p.r : p.k) + base;
    const uint16_t* const val = (REV ? p.gy : p.v) + base;
    float pw[CT][8], dec[CT][4];
    auto log_decay = [&](int j) __attribute__((always_inline)) { return -expf(bf2f(p.w[h * HN + j])); };
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int j0 = 16 * (CT * q + ct);
        const float l = log_decay(j0 + l16);
#pragma unroll
        for (int e = 0; e < 8; ++e) pw[ct][e] = wpow(l, REV ? slot_token(g, e) : 31 - slot_token(g, e));
#pragma unroll
        for (int v = 0; v < 4; ++v) dec[ct][v] = REV ? wpow(l, L) : wpow(log_decay(j0 + 4 * g + v), L);
    }
    uint4 x[2][NP];
    auto fetch = [&](const int i) __attribute__((always_inline)) {       // i-th chunk in the direction of travel
        const int c = REV ? max(chunks - 1 - i, 0) : min(i, chunks - 1);
        const rows_t kr = rows_of(key + static_cast<size_t>(c) * L * C, left - c * L, C), vr = rows_of(val + static_cast<size_t>(c) * L * C, left - c * L, C);
#pragma unroll
        for (int z = 0; z < NP; ++z) {
            const int lo = 2 * ((row0 + z * A::ROWS) * C + c8);
            x[0][z] = load16(kr, lo); x[1][z] = load16(vr, lo);
        }
    };
    auto put = [&](const int set) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < NP; ++z) {
            const lds_t o = sb + set * 2 * A::PLANE + (row0 + z * A::ROWS) * A::ROW + 2 * c8;
            lds_st<bf16x8>(o, op4(x[0][z])); lds_st<bf16x8>(o + A::PLANE, op4(x[1][z]));
        }
    };
    f32x4 acc[CT][NT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < NT; ++e) acc[ct][e] = ZERO4;
    fetch(0);
    put(0);
    fetch(1);
    __syncthreads();
    for (int i = 0; i < chunks; ++i) {
        lds_t o = sb + (i & 1) * 2 * A::PLANE + (4 * g + (l16 >> 2)) * A::ROW + 8 * (l16 & 3);
        opaque(o);
        Op2 k[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) k[ct] = scaled(ld_tra<A::ROW>(o + 32 * (CT * q + ct)), pw[ct]);
#pragma unroll
        for (int e = 0; e < NT; ++e) {
            const bf16x8 v = ld_tra<A::ROW>(o + A::PLANE + 32 * e);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                f32x4 s = acc[ct][e];
#pragma unroll
                for (int t = 0; t < 4; ++t) s[t] *= dec[ct][t];
                acc[ct][e] = REV ? mfma(v, k[ct].l, mfma(v, k[ct].h, s)) : mfma(k[ct].l, v, mfma(k[ct].h, v, s));
            }
        }
        put((i + 1) & 1);
        fetch(i + 2);
        __syncthreads();
    }
    float* const out = p.local + (static_cast<size_t>(rel) * (p.NB - 1) + m) * HN * HN;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < NT; ++e) {
            const int j0 = 16 * (CT * q + ct), i0 = 16 * e;
            *reinterpret_cast<f32x4*>(out + (REV ? (j0 + l16) * HN + i0 + 4 * g : (i0 + l16) * HN + j0 + 4 * g)) = acc[ct][e];
        }
}

// ---------------------------------------------------------------------------------------------------- forward
// Waves 0..3 hold St[ct][jt][v] = S[j = 16 jt + 4 g + v][i = own], as it stands the B operand of a contraction over j.  Waves 4..7
// load (two chunks ahead of the planes, the planes two chunks ahead of their use) and make the next chunk's tile in parts of 32
// key channels.  One barrier a chunk.
// Planes: R' = r o^{t-16}, K' = k o^{15-t} (they serve the tile, the state times o^16 on its way in and out of the update); RAW, for
// strong decays: r o^t, k o^{31-t}, and the tile is made from the raw rows (read once more, from L2).
template <int HN, bool RAW> DEVINL void fwd_states(const ArgsW& p, lds_t sb, int q, int lane, const Part& part) {
    using A = G<HN>;
    constexpr int CT = A::CT, KS = A::KS, NJ = A::NB16;
    const int l16 = lane & 15, g = lane >> 4, T = part.left, C = p.C, nch = part.chunks;
    const size_t base = part.base;
    float dd[NJ][4];                                     // o^16; RAW: o^32
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt)
#pragma unroll
        for (int v = 0; v < 4; ++v) dd[jt][v] = wpow(lds_f(sb + A::LAM + 4 * (16 * jt + 4 * g + v)), RAW ? 32 : 16);
    f32x4 St[CT][NJ];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int jt = 0; jt < NJ; ++jt) St[ct][jt] = ZERO4;
    if (part.n > 0) {                                    // the state that enters the block, from what the blocks before leave
        const float* x = p.local + static_cast<size_t>(part.rel) * (p.NB - 1) * HN * HN + (16 * CT * q + l16) * HN + 4 * g;
#pragma unroll 2
        for (int m = 0; m < part.n; ++m, x += HN * HN)
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) {
                const f32x4 d = lds_ld<f32x4>(sb + A::BLK + 4 * (16 * jt + 4 * g));
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) St[ct][jt] = St[ct][jt] * d + *reinterpret_cast<const f32x4*>(x + 16 * ct * HN + 16 * jt);
            }
    }
    float* const sv = p.saved != nullptr ? saved_state<HN>(p, part) + 16 * CT * q + l16 + 4 * g * HN : nullptr;
    uint16_t* const out = p.y + base + 16 * CT * q;
    const int to = tile_offset(l16, g, C);
    const lds_t orow = sb + A::BASE + l16 * A::ROW + 8 * g, otr = sb + A::BASE + (4 * g + (l16 >> 2)) * A::ROW + 8 * (l16 & 3);
    __syncthreads();                                     // chunks 0 and 1 are there
    __syncthreads();                                     // and the first tile
    int sl = 0;
    for (int c = 0; c < nch; ++c) {
        lds_t xr = orow + sl * A::FSLOT, xt = otr + sl * A::FSLOT;
        opaque(xr); opaque(xt);
        sl = sl == 2 ? 0 : sl + 1;
        // (past the caches at 128 channels a head, where they are half of what is written: forward and backward at B=8, T=4096, C=4096 take 1437 us
        // and 1427 so, 1482 and 1467 on another machine; at 64 channels 566 and 569.  The backward's reads of them past the caches: 1454 and 1515.)
        if (sv != nullptr && (c & 1) == 0) {
            float* const d = sv + static_cast<size_t>(c >> 1) * HN * HN;
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        if constexpr (HN == 128) __builtin_nontemporal_store(St[ct][jt][v], &d[(16 * jt + v) * HN + 16 * ct]);
                        else d[(16 * jt + v) * HN + 16 * ct] = St[ct][jt][v];
                    }
        }
        f32x4 Y[2][CT];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) Y[tt][ct] = ZERO4;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            Op2 x[2];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                x[tt].h = ld_acc(xr + A::FRH + 16 * tt * A::ROW + 64 * ks);
                x[tt].l = ld_acc(xr + A::FRL + 16 * tt * A::ROW + 64 * ks);
            }
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                if constexpr (!RAW) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) { St[ct][2 * ks][v] *= dd[2 * ks][v]; St[ct][2 * ks + 1][v] *= dd[2 * ks + 1][v]; }
                }
                const Op2 s = split8(St[ct][2 * ks], St[ct][2 * ks + 1]);
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) Y[tt][ct] = mm3(x[tt], s, Y[tt][ct]);
            }
        }
        bf16x8 vo[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) vo[ct] = ld_tra<A::ROW>(xt + A::FV + 32 * (CT * q + ct));
        Op2 at[2];
        take_parts<A::PARTS, A::PART>(sb + A::FPART + (c & 1) * (A::PARTS * A::PART), lane, at);
        const rows_t o = rows_of(out + static_cast<size_t>(c) * L * C, T - c * L, C);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const f32x4 y = mfma(at[tt].l, vo[ct], mfma(at[tt].h, vo[ct], Y[tt][ct]));
                store_tile(o, to + 32 * tt * C + 32 * ct, C, l16, y);
            }
#pragma unroll
        for (int jt = 0; jt < NJ; ++jt) {
            const bf16x8 kh = ld_tra<A::ROW>(xt + A::FKH + 32 * jt), kl = ld_tra<A::ROW>(xt + A::FKL + 32 * jt);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                f32x4 s = St[ct][jt];
                if constexpr (RAW) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) s[v] *= dd[jt][v];
                }
                s = mfma(kl, vo[ct], mfma(kh, vo[ct], s));
                if constexpr (!RAW) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) s[v] *= dd[jt][v];
                }
                St[ct][jt] = s;
            }
        }
        __syncthreads();
    }
}

template <int HN, bool RAW> DEVINL void fwd_loads(const ArgsW& p, lds_t sb, int tp, const Part& part) {
    using A = G<HN>;
    constexpr int NP = A::PASSES;
    const int lane = tp & 63, q = tp >> 6, l16 = lane & 15, g = lane >> 4, T = part.left, C = p.C, nch = part.chunks;
    const size_t base = part.base;
    const int row0 = tp / A::PIECES, c8 = (tp % A::PIECES) * 8;
    float u[8], pr[NP][8], pk[NP][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float l = lds_f(sb + A::LAM + 4 * (c8 + e));
        u[e] = lds_f(sb + A::U + 4 * (c8 + e));
#pragma unroll
        for (int z = 0; z < NP; ++z) {
            const int t = row0 + z * A::ROWS;
            pr[z][e] = wpow(l, RAW ? t : t - 16);
            pk[z][e] = wpow(l, RAW ? 31 - t : 15 - t);
        }
    }
    [[maybe_unused]] TilePowers tpw;
    if constexpr (RAW) tile_powers(tpw, sb + A::LAM + 4 * (32 * (q % A::PARTS) + 8 * g), l16);
    uint4 x[2][3][NP];
    auto fetch = [&](const int c, uint4 (&d)[3][NP]) __attribute__((always_inline)) {
        const int cc = min(c, nch - 1);                  // (the same loads in every iteration)
        const size_t o = base + static_cast<size_t>(cc) * L * C;
        const int left = T - c * L;
        const rows_t r = rows_of(p.r + o, left, C), k = rows_of(p.k + o, left, C), v = rows_of(p.v + o, left, C);
#pragma unroll
        for (int z = 0; z < NP; ++z) {
            const int lo = 2 * ((row0 + z * A::ROWS) * C + c8);
            d[0][z] = load16(r, lo); d[1][z] = load16(k, lo); d[2][z] = load16(v, lo);
        }
    };
    auto put = [&](const int sl, const uint4 (&d)[3][NP]) __attribute__((always_inline)) {
        const lds_t s = sb + A::BASE + sl * A::FSLOT;
#pragma unroll
        for (int z = 0; z < NP; ++z) {
            const int t = row0 + z * A::ROWS;
            float r[8], k[8], a = 0.f;
            unpack8(d[0][z], r); unpack8(d[1][z], k);
#pragma unroll
            for (int e = 0; e < 8; ++e) { a = fmaf(r[e] * u[e], k[e], a); r[e] *= pr[z][e]; k[e] *= pk[z][e]; }
            const Op2 ro = split8(r), ko = split8(k);
            const lds_t o = s + t * A::ROW + 2 * c8;
            lds_st<bf16x8>(o + A::FRH, ro.h); lds_st<bf16x8>(o + A::FRL, ro.l);
            lds_st<bf16x8>(o + A::FKH, ko.h); lds_st<bf16x8>(o + A::FKL, ko.l);
            lds_st<bf16x8>(o + A::FV, op4(d[2][z]));
            a = lanes_sum<A::PIECES>(a);
            if (c8 == 0) lds_st<float>(s + A::FRUK + 4 * t, a);
        }
    };
    auto tile = [&](const int c, const int sl) __attribute__((always_inline)) {
        if (q >= A::PARTS) return;
        f32x4 qd[3];
        const lds_t s = sb + A::BASE + sl * A::FSLOT;
        if constexpr (RAW) {
            const size_t co = base + static_cast<size_t>(c) * L * C;
            const rows_t rr = rows_of(p.r + co, T - c * L, C), kk = rows_of(p.k + co, T - c * L, C);
            bf16x8 r[2], k[2];
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const int o = 2 * ((16 * z + l16) * C + 32 * q + 8 * g);
                r[z] = op4(load16(rr, o)); k[z] = op4(load16(kk, o));
            }
            raw_part(r, k, tpw, qd);
        } else {
            Op2 xo[2], yo[2];
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const lds_t o = s + (16 * z + l16) * A::ROW + 64 * q + 16 * g;
                xo[z] = {ld_op(o + A::FRH), ld_op(o + A::FRL)};
                yo[z] = {ld_op(o + A::FKH), ld_op(o + A::FKL)};
            }
#pragma unroll
            for (int z = 0; z < 3; ++z) qd[z] = mm3(yo[Quad<true>::ROWT[z]], xo[Quad<true>::LANET[z]], ZERO4);
        }
        const float diag[2] = {q == 0 ? lds_f(s + A::FRUK + 4 * l16) : 0.f, q == 0 ? lds_f(s + A::FRUK + 4 * (16 + l16)) : 0.f};
        const lds_t out = sb + A::FPART + ((c & 1) * A::PARTS + q) * A::PART;
        put_quad<true, 0>(out, qd[0], diag[0], lane); put_quad<true, 1>(out, qd[1], 0.f, lane); put_quad<true, 2>(out, qd[2], diag[1], lane);
    };
    fetch(0, x[0]); fetch(1, x[1]);
    put(0, x[0]); fetch(2, x[0]);
    put(1, x[1]); fetch(3, x[1]);
    __syncthreads();
    tile(0, 0);
    __syncthreads();
    int sl = 2;
    for (int c0 = 0; c0 < nch; c0 += 2) {
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const int c = c0 + z;
            if (c >= nch) break;
            put(sl, x[z]);
            fetch(c + 4, x[z]);
            if (c + 1 < nch) tile(c + 1, sl == 0 ? 2 : sl - 1);
            sl = sl == 2 ? 0 : sl + 1;
            __syncthreads();
        }
    }
}

template <int HN>
__global__ __launch_bounds__(NTH, 2) void wkv5b_fwd(const ArgsW p) {
    const lds_t sb = lds_of(smem_raw);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Part part = part_of(p, HN, false);
    if (HN == 64 && !strong_layer(p.w, p.C, tid & 63)) return;      // the one-sweep kernels of wkv6 have done this layer
    const float lmin = head_setup<HN>(p, sb, part, tid);            // (the decays of every head go to p.decay)
    if (steps_head<false, HN>(p.w, nullptr, part.h * HN)) return;
    __syncthreads();
    if (w < 4) {
        if (lmin < LAM_MID) fwd_states<HN, true>(p, sb, w, tid & 63, part);
        else fwd_states<HN, false>(p, sb, w, tid & 63, part);
    } else {
        if (lmin < LAM_MID) fwd_loads<HN, true>(p, sb, tid - 256, part);
        else fwd_loads<HN, false>(p, sb, tid - 256, part);
    }
}

// ---------------------------------------------------------------------------------------------------- backward
// One reverse sweep, two barriers a chunk, two roles of HN / 16 waves each (head size 128: all sixteen of a CU):
//   D (16 key channels j): the gradient state dS[ib][v] = D[i = 16 ib + 4 g + v][j = own], the B operand of contractions over the
//      value channel: gk in the first half of a chunk; gr, the gradient state's update and the decay gradient in the second.
//      The saved state passes through in tiles (an odd chunk's is one update away from the saved one, made on the way).
//   E (32 value channels i of 16 tokens): first half: the loads, the rows of the next chunk to LDS, this chunk's tile A in parts (a
//      wave makes the quadrants within the halves or the one across, of 32 channels); second half: gv, for which the D waves left
//      their gradient state in LDS (hi, lo) in the first, and the next chunk's tile B as the operands that the D waves take: B and
//      its weighted form with lane = source, its transpose with lane = sink.
// Twice four waves, of 32 key channels each and with the tile B made by each of the D waves, took 1042 us (B8 T4096 C4096 N128) where
// these take 986 (heads of 64: the same), with the same bits: every sum has that kernel's order, so gr's tile part is kept over the barrier and
// its bonus term added after the state's (the other way round 981 us).  Without its memory operations the kernel takes 753 us, and its 3.3 GB
// about 660 at a copy's rate.
template <bool LANE_SNK> DEVINL void mask(f32x4 (&b)[3], int l16, int g) {
#pragma unroll
    for (int z = 0; z < 3; ++z)
#pragma unroll
        for (int v = 0; v < 4; ++v) b[z][v] = causal<LANE_SNK>(z, l16, 4 * g + v) ? b[z][v] : 0.f;
}
// The tile B as operands of its lane tiles, 3 KB a form.  The lane tile that meets both halves of the other side takes 16 bytes a lane
// and term; the other one has zeros on one side (HIGH: in its low slots), the two terms share 16 bytes.  LAGS: every element times
// the tokens between, lag + 16 (row tile - lane tile) + v.
template <bool LANE_SNK, bool LAGS> DEVINL void put_tile(lds_t o, const f32x4 (&t)[3], int lane, float lag = 0.f) {
    const auto two = [&](int z, int v) __attribute__((always_inline)) {
        const float m = lag + static_cast<float>(16 * (Quad<LANE_SNK>::ROWT[z] - Quad<LANE_SNK>::LANET[z]) + v);
        return LAGS ? hilo2p(t[z][v], m, t[z][v + 1], m + 1.f) : hilo2k(t[z][v], t[z][v + 1]);
    };
    constexpr int full = LANE_SNK ? 1 : 0, half = LANE_SNK ? 0 : 2;
    const HL a = two(full, 0), b = two(full, 2), c = two(full + 1, 0), d = two(full + 1, 2), e = two(half, 0), f = two(half, 2);
    o += 16 * lane;
    lds_st<bf16x8>(o, as_op(a.h, b.h, c.h, d.h)); lds_st<bf16x8>(o + 1024, as_op(a.l, b.l, c.l, d.l));
    lds_st<u32x4>(o + 2048, u32x4{e.h, f.h, e.l, f.l});
}
template <bool HIGH> DEVINL Op2 half_op(lds_t o) {
    const u32x4 x = lds_ld<u32x4>(o + 2048);
    return HIGH ? Op2{as_op(0u, 0u, x[0], x[1]), as_op(0u, 0u, x[2], x[3])} : Op2{as_op(x[0], x[1], 0u, 0u), as_op(x[2], x[3], 0u, 0u)};
}
DEVINL Op2 full_op(lds_t o) { return {ld_op(o), ld_op(o + 1024)}; }

// The lane's number, worked out where it is used.  (What is derived from threadIdx is kept in registers across the chunk loop, and where
// those do not last, in scratch: a reload waits for all loads under way.)
DEVINL uint32_t lane_now() {
    uint32_t all = ~0u;
    asm volatile("" : "+s"(all));
    return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u));
}

template <int HN> DEVINL void role_d(const ArgsW& p, lds_t sb, int q, int lane, const Part& part) {
    using A = G<HN>;
    constexpr int KS = A::KS, NI = A::NB16;
    const int l16 = lane & 15, g = lane >> 4, T = part.left, C = p.C, nch = part.chunks;
    const size_t base = part.base;
    // Powers of a set of eight slots, token 16 a + 4 g + b: a base per lane times o^b times o^{16 a} (or the reverse); the eight would
    // take the registers that the states need.  Bases: cb of o^{t-m}, kb of o^{m-1-t}, m the middle of the token's half.
    const float l = lds_f(sb + A::LAM + 4 * (16 * q + l16));
    const float o1 = wpow(l, 1), o2 = wpow(l, 2), o3 = wpow(l, 3), o8 = wpow(l, 8), o16 = wpow(l, 16), o32 = wpow(l, 32);
    const float cb = wpow(l, 4 * g - 8), kb = wpow(l, 4 - 4 * g);
    f32x4 dS[NI];
#pragma unroll
    for (int ib = 0; ib < NI; ++ib) dS[ib] = ZERO4;
    if (part.n + 1 < p.NB) {                             // the gradient of the state that leaves the block, from what the blocks after take up
        const float* x = p.local + (static_cast<size_t>(part.rel) * (p.NB - 1) + p.NB - 2) * HN * HN + (16 * q + l16) * HN + 4 * g;
        const float d = lds_f(sb + A::BLK + 4 * (16 * q + l16));
#pragma unroll 1
        for (int m = p.NB - 1; m > part.n; --m, x -= HN * HN)
#pragma unroll
            for (int ib = 0; ib < NI; ++ib) dS[ib] = dS[ib] * d + *reinterpret_cast<const f32x4*>(x + 16 * ib);
    }
    float gw = 0.f, gP = 0.f, gu = 0.f;
    // (hidden: hoisted out of the loop the powers and token numbers would take registers all the same)
    auto hide = [](float x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); return x; };
    auto up = [&](float base, bool span, float (&f)[8]) __attribute__((always_inline)) {
        base = hide(base);
        f[0] = base; f[1] = base * o1; f[2] = base * o2; f[3] = base * o3;
#pragma unroll
        for (int e = 0; e < 4; ++e) f[4 + e] = span ? f[e] * o16 : f[e];
    };
    auto down = [&](float base, bool span, float (&f)[8]) __attribute__((always_inline)) {
        base = hide(base);
        f[4] = base * o3; f[5] = base * o2; f[6] = base * o1; f[7] = base;
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = span ? f[4 + e] * o16 : f[4 + e];
    };
    auto to_ref = [&](float (&f)[8]) __attribute__((always_inline)) { up(cb, false, f); };                    // o^{t-m}
    auto from_ref = [&](float (&f)[8]) __attribute__((always_inline)) { down(kb, false, f); };                // o^{m-1-t}
    auto from_start = [&](float (&f)[8]) __attribute__((always_inline)) { up(hide(cb) * o8, true, f); };            // o^t
    auto to_end = [&](float (&f)[8]) __attribute__((always_inline)) { down(hide(kb) * o8, true, f); };              // o^{31-t}
    auto stage = [] __attribute__((always_inline)) () { __builtin_amdgcn_sched_barrier(0); };      // (or operands are asked for so early that the registers do not hold them)
    // The operands that a tile's lane tiles 0 and 1 are applied to, referred to the middle of the lane's half whichever half a slot's
    // token lies in.  f: the powers of the token in its own half.  Only the far pair (sinks of the second half for a source of the
    // first, or sources of the first for a sink of the second) takes o^16; the slots on the wrong side of the lane tile meet zeros.
    auto tile_operands = [&](bool sinks, const bf16x8& x, const float (&f)[8], Op2 (&o)[2]) __attribute__((always_inline)) {
        float fx[8], ff[4];
        unpack(x, fx);
#pragma unroll
        for (int e = 0; e < 8; ++e) fx[e] *= f[e];
        o[0] = o[1] = split8(fx);
#pragma unroll
        for (int e = 0; e < 4; ++e) ff[e] = (sinks ? fx[4 + e] : fx[e]) * o8 * o8;      // (o^16 may underflow where this does not)
        const HL a = hilo2k(ff[0], ff[1]), b = hilo2k(ff[2], ff[3]);
        Op2& w = o[sinks ? 0 : 1];
        const uint4 h = __builtin_bit_cast(uint4, w.h), lo = __builtin_bit_cast(uint4, w.l);
        w = sinks ? Op2{as_op(h.x, h.y, a.h, b.h), as_op(lo.x, lo.y, a.l, b.l)} : Op2{as_op(a.h, b.h, h.z, h.w), as_op(a.l, b.l, lo.z, lo.w)};
    };
    const float* const sv = saved_state<HN>(p, part);
    auto fetch_state = [&](int c, int ks, uint32_t so, f32x4 (&s)[2]) __attribute__((always_inline)) {      // (a scalar base and one lane offset)
        const char* const d = reinterpret_cast<const char*>(sv + static_cast<size_t>(c >> 1) * HN * HN + 32 * ks);
#pragma unroll
        for (int z = 0; z < 2; ++z) s[z] = *reinterpret_cast<const f32x4*>(d + 64 * z + so);
    };
    // the lane's addresses, anew in each half of a chunk
    struct Lane { lds_t row, tra, tile; uint32_t state; int out; float t; };
    auto lane_of = [&]() __attribute__((always_inline)) {
        const uint32_t me = lane_now(), n = me & 15, gg = me >> 4;
        return Lane{n * A::ROW + 8 * gg, (4 * gg + (n >> 2)) * A::ROW + 8 * (n & 3), 16 * me, ((16 * q + n) * HN + 4 * gg) * 4,
                    tile_offset(static_cast<int>(n), static_cast<int>(gg), C), static_cast<float>(4 * gg)};
    };
    // second half of a chunk: gr, update
    auto second = [&](auto odd_, const int c, const f32x4 (&tx)[2], f32x4 (&Sn)[2][2]) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd_)::value;
        const lds_t sx = sb + A::BASE + (ODD ? A::SLOT : 0);
        const Lane at = lane_of();
        const lds_t xr = at.row + sx, xu = at.tra + sx, xt = xu + 32 * q, qt = at.tra + sb + A::BASE + (ODD ? 0 : A::SLOT), xs = sx + 4 * static_cast<lds_t>(at.t);
        const rows_t gr_ = rows_of(p.gr + base + static_cast<size_t>(c) * L * C + 16 * q, T - c * L, C);
        Op2 rs, kp;
        {
            float f[8];
            from_start(f);
            rs = scaled(ld_tra<A::ROW>(xt + A::R), f);
            stage();
            if constexpr (ODD) {
                to_end(f);
                kp = scaled(ld_tra<A::ROW>(qt + A::K + 32 * q), f);
            }
        }
        f32x4 X[2] = {ZERO4, ZERO4};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const bf16x8 gt = ld_tra<A::ROW>(xu + A::GY + 64 * ks + 32 * z);
                bf16x8 vt;
                if constexpr (ODD) vt = ld_tra<A::ROW>(qt + A::V + 64 * ks + 32 * z);
                f32x4& s = Sn[ks & 1][z];
                f32x4& d = dS[2 * ks + z];
                if constexpr (ODD) s = mfma(vt, kp.l, mfma(vt, kp.h, s * o32));
                gP += (s[0] * d[0] + s[1] * d[1]) + (s[2] * d[2] + s[3] * d[3]);
                d = mfma(gt, rs.l, mfma(gt, rs.h, d * o32));
                stage();
            }
            const Op2 s = split8(Sn[ks & 1][0], Sn[ks & 1][1]);
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const bf16x8 ga = ld_acc(xr + A::GY + 16 * z * A::ROW + 64 * ks);
                X[z] = mfma(ga, s.l, mfma(ga, s.h, X[z]));
            }
            if (ks + 2 < KS) fetch_state(c, ks + 2, at.state, Sn[ks & 1]);
            stage();
        }
        stage();
        {
            const uint4 r4 = __builtin_bit_cast(uint4, ld_tra<A::ROW>(xt + A::R)), k4 = __builtin_bit_cast(uint4, ld_tra<A::ROW>(xt + A::K));
            const float u = lds_f(sb + A::U + 64 * q + (at.tile >> 2 & 60u));
            const float bc = hide(cb), bs = bc * o8;
            const float pc[4] = {bc, bc * o1, bc * o2, bc * o3}, ps[4] = {bs, bs * o1, bs * o2, bs * o3};
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const f32x4 vg4 = lds_ld<f32x4>(xs + A::VG + 64 * z);
                const uint32_t rw[2] = {z ? r4.z : r4.x, z ? r4.w : r4.y}, kw[2] = {z ? k4.z : k4.x, z ? k4.w : k4.y};
                const float th = at.t + static_cast<float>(16 * z);
                f32x4 o;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float r = v & 1 ? bf_hi(rw[v >> 1]) : bf_lo(rw[v >> 1]), k = v & 1 ? bf_hi(kw[v >> 1]) : bf_lo(kw[v >> 1]);
                    const float x = X[z][v] * (z ? ps[v] * o16 : ps[v]);
                    gw = fmaf(r * (th + static_cast<float>(v)), x, gw);
                    o[v] = fmaf(k * vg4[v], u, fmaf(tx[z][v], pc[v], x));
                }
                store_tile(gr_, at.out + 32 * z * C, C, static_cast<int>(at.tile >> 4), o);
                stage();
            }
        }
    };
    auto chunk = [&](auto odd_, const int c) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd_)::value;
        const lds_t sx = sb + A::BASE + (ODD ? A::SLOT : 0);
        const Lane at = lane_of();
        const lds_t xr = at.row + sx, xt = at.tra + sx + 32 * q, xs = sx + 4 * static_cast<lds_t>(at.t), ho = at.row + sb + A::DSH + 16 * q * A::ROW, tl = at.tile + sb + A::BTILE;
        const size_t co = base + static_cast<size_t>(c) * L * C + 16 * q;
        const rows_t gk_ = rows_of(p.gk + co, T - c * L, C);
        // ---- first half: gk, gr's tile part
        f32x4 Z[2] = {ZERO4, ZERO4};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const Op2 s = split8(dS[2 * ks], dS[2 * ks + 1]);
            const uint4 hi = __builtin_bit_cast(uint4, s.h), lo = __builtin_bit_cast(uint4, s.l);
            const lds_t o = ho + 64 * ks;
            lds_st<u32x2>(o, u32x2{hi.x, hi.y}); lds_st<u32x2>(o + 32, u32x2{hi.z, hi.w});
            lds_st<u32x2>(o + (A::DSL - A::DSH), u32x2{lo.x, lo.y}); lds_st<u32x2>(o + (A::DSL - A::DSH) + 32, u32x2{lo.z, lo.w});
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const bf16x8 va = ld_acc(xr + A::V + 16 * z * A::ROW + 64 * ks);
                Z[z] = mfma(va, s.l, mfma(va, s.h, Z[z]));
            }
        }
        f32x4 tx[2];                                     // gr's tile part
        {
            const bf16x8 rT = ld_tra<A::ROW>(xt + A::R), kT = ld_tra<A::ROW>(xt + A::K);
            const uint4 r4 = __builtin_bit_cast(uint4, rT), k4 = __builtin_bit_cast(uint4, kT);
            const float u = lds_f(sb + A::U + 64 * q + (at.tile >> 2 & 60u));
            Op2 ro[2];
            {
                float pm[8];
                to_ref(pm);
                tile_operands(true, rT, pm, ro);
            }
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                f32x4 tz, tw;
                if (z) { tz = mm3(half_op<true>(tl), ro[z], ZERO4); tw = mm3(half_op<true>(tl + 3072), ro[z], ZERO4); }
                else { tz = mm3(full_op(tl), ro[z], ZERO4); tw = mm3(full_op(tl + 3072), ro[z], ZERO4); }
                const f32x4 vg4 = lds_ld<f32x4>(xs + A::VG + 64 * z);
                const uint32_t rw[2] = {z ? r4.z : r4.x, z ? r4.w : r4.y}, kw[2] = {z ? k4.z : k4.x, z ? k4.w : k4.y};
                const float th = at.t + static_cast<float>(16 * z), ba = hide(kb), be = ba * o8;
                const float pf[4] = {ba * o3, ba * o2, ba * o1, ba}, pe[4] = {be * o3, be * o2, be * o1, be};
                f32x4 o;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float r = v & 1 ? bf_hi(rw[v >> 1]) : bf_lo(rw[v >> 1]), k = v & 1 ? bf_hi(kw[v >> 1]) : bf_lo(kw[v >> 1]);
                    const float zs = Z[z][v] * (z == 0 ? pe[v] * o16 : pe[v]), t = th + static_cast<float>(v), rv = r * vg4[v];
                    gw = fmaf(k, fmaf(zs, 31.f - t, tw[v] * pf[v]), gw);
                    gu = fmaf(rv, k, gu);
                    o[v] = fmaf(rv, u, fmaf(tz[v], pf[v], zs));
                }
                store_tile(gk_, at.out + 32 * z * C, C, static_cast<int>(at.tile >> 4), o);
            }
            {
                float pm[8];
                Op2 ko[2];
                from_ref(pm);
                tile_operands(false, kT, pm, ko);
                tx[0] = mm3(half_op<false>(tl + 2 * 3072), ko[0], ZERO4);
                tx[1] = mm3(full_op(tl + 2 * 3072), ko[1], ZERO4);
            }
        }
        f32x4 Sn[2][2];
        fetch_state(c, 0, at.state, Sn[0]);
        fetch_state(c, 1, at.state, Sn[1]);
        __syncthreads();                                 // the rows of the chunk before are there, the gradient state is handed over
        second(odd_, c, tx, Sn);
        __syncthreads();
    };
    __syncthreads();                                     // the top chunk is there
    __syncthreads();                                     // and its tile B
    for (int c = nch - 1; c >= 0; c -= 2) {
        chunk(std::true_type{}, c);
        chunk(std::false_type{}, c - 1);
    }
    const size_t o = (static_cast<size_t>(part.n) * p.heads + part.rel) * HN + 16 * q + l16;
    const float sw = allreduce_rows(fmaf(32.f * o32, gP, gw)), su = allreduce_rows(gu);
    if (g == 0) {
        if (p.NB > 1) { p.gw32[o] = l * sw; p.gu32[o] = su; }
        else { p.gw[o] = f2bf(l * sw); p.gu[o] = f2bf(su); }      // (a launch of whole sequences begins with head 0)
    }
}

template <int HN> DEVINL void role_e(const ArgsW& p, lds_t sb, int te, const Part& part_) {
    using A = G<HN>;
    constexpr int KS = A::KS, PARTS = A::PARTS;
    const int w = __builtin_amdgcn_readfirstlane(te >> 6), lane = te & 63, l16 = lane & 15, g = lane >> 4, T = part_.left, C = p.C, nch = part_.chunks;
    const size_t base = part_.base;
    const int row0 = te / A::PIECES, c8 = (te % A::PIECES) * 8;
    // gv: value channels 32 wq .. + 31, tokens 16 wz .. + 15; tile A: channels 32 part .., the quadrant across the halves or the others
    const int wq = w >> 1, wz = w & 1, part = w % PARTS;
    const bool across = w >= PARTS;
    const int form = PARTS > 2 ? w - PARTS : (w == 0 ? 1 : (w == 1 ? -1 : 2 * (w - 2)));       // of tile B: 0 as it is, 1 weighted, 2 transposed
    float cke[KS][8];                                    // o^{31-t} of token 16 wz + l16, channel 32 ks + 8 g + e
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) cke[ks][e] = wpow(lds_f(sb + A::LAM + 4 * (32 * ks + 8 * g + e)), 31 - 16 * wz - l16);
    float px[8], py[8];                                  // tile A: as sink and as source, see TilePowers
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float l = lds_f(sb + A::LAM + 4 * (32 * part + 8 * g + e));
        px[e] = wpow(l, across ? l16 : l16 - 8); py[e] = wpow(l, across ? 15 - l16 : 7 - l16);
    }
    auto fetch = [&](const int c, uint4 (&d)[4]) __attribute__((always_inline)) {
        const int cc = max(c, 0);
        const size_t o = base + static_cast<size_t>(cc) * L * C;
        const int left = T - cc * L, lo = 2 * (row0 * C + c8);
        const rows_t r = rows_of(p.r + o, left, C), k = rows_of(p.k + o, left, C), v = rows_of(p.v + o, left, C), gy = rows_of(p.gy + o, left, C);
        d[0] = load16(r, lo); d[1] = load16(k, lo); d[2] = load16(v, lo); d[3] = load16(gy, lo);
    };
    auto put = [&](const int sl, const uint4 (&d)[4]) __attribute__((always_inline)) {
        const lds_t s = sb + A::BASE + sl * A::SLOT;
        const f32x4 u[2] = {lds_ld<f32x4>(sb + A::U + 4 * c8), lds_ld<f32x4>(sb + A::U + 4 * c8 + 16)};      // (registers for these across the loop would spill others)
        const lds_t o = s + row0 * A::ROW + 2 * c8;
#pragma unroll
        for (int i = 0; i < 4; ++i) lds_st<bf16x8>(o + i * A::PLANE, op4(d[i]));
        float r[8], k[8], v[8], gy[8], a = 0.f, b = 0.f;
        unpack8(d[0], r); unpack8(d[1], k); unpack8(d[2], v); unpack8(d[3], gy);
#pragma unroll
        for (int e = 0; e < 8; ++e) { a = fmaf(r[e] * u[e >> 2][e & 3], k[e], a); b = fmaf(v[e], gy[e], b); }
        a = lanes_sum<A::PIECES>(a); b = lanes_sum<A::PIECES>(b);
        if (c8 == 0) { lds_st<float>(s + A::RUK + 4 * row0, a); lds_st<float>(s + A::VG + 4 * row0, b); }
    };
    // the three forms of tile B of the chunk in a slot, one a wave, by those that have less to do for tile A before others
    auto tile_b = [&](const int sl) __attribute__((always_inline)) {
        if (form < 0 || form > 2) return;
        const int lane = static_cast<int>(lane_now()), l16 = lane & 15, g = lane >> 4;
        lds_t xr = sb + A::BASE + sl * A::SLOT + l16 * A::ROW + 8 * g;
        opaque(xr);
        const lds_t out = sb + A::BTILE;
        f32x4 t[3] = {ZERO4, ZERO4, ZERO4};
        const auto products = [&](auto transposed_, const lds_t rows, const lds_t cols) __attribute__((always_inline)) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const bf16x8 a[2] = {ld_acc(rows + 64 * ks), ld_acc(rows + 16 * A::ROW + 64 * ks)}, b[2] = {ld_acc(cols + 64 * ks), ld_acc(cols + 16 * A::ROW + 64 * ks)};
                using Q = Quad<decltype(transposed_)::value>;
#pragma unroll
                for (int z = 0; z < 3; ++z) t[z] = mfma(a[Q::ROWT[z]], b[Q::LANET[z]], t[z]);
            }
        };
        if (form == 2) {
            products(std::true_type{}, xr + A::V, xr + A::GY);
            mask<true>(t, l16, g);
            put_tile<true, false>(out + 2 * 3072, t, lane);
            return;
        }
        products(std::false_type{}, xr + A::GY, xr + A::V);
        mask<false>(t, l16, g);
        if (form == 0) put_tile<false, false>(out, t, lane);
        else put_tile<false, true>(out + 3072, t, lane, static_cast<float>(4 * g - (l16 + 1)));       // for the decay gradient
    };
    uint4 next[4];                                       // a chunk ahead of its way to LDS
    fetch(nch - 1, next);
    put(1, next);
    fetch(nch - 2, next);
    auto chunk = [&](auto odd_, const int c) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd_)::value;
        constexpr int PREV = ODD ? 0 : 1;
        const lds_t sx = sb + A::BASE + (ODD ? A::SLOT : 0);
        // ---- first half
        {
            const int lane = static_cast<int>(lane_now()), l16 = lane & 15, g = lane >> 4;
            lds_t o = sx + l16 * A::ROW + 64 * part + 16 * g;
            opaque(o);
            const lds_t out = sb + A::BPART + part * A::PART;
            if (across) {
                const Op2 x = scaled(ld_op(o + A::R + 16 * A::ROW), px), y = scaled(ld_op(o + A::K), py);
                put_quad<false, 1>(out, mm3(x, y, ZERO4), 0.f, lane);
            } else {
#pragma unroll
                for (int z = 0; z < 2; ++z) {
                    const Op2 x = scaled(ld_op(o + A::R + 16 * z * A::ROW), px), y = scaled(ld_op(o + A::K + 16 * z * A::ROW), py);
                    const float diag = part == 0 ? lds_f(sx + A::RUK + 4 * (16 * z + l16)) : 0.f;
                    if (z == 0) put_quad<false, 0>(out, mm3(x, y, ZERO4), diag, lane);
                    else put_quad<false, 2>(out, mm3(x, y, ZERO4), diag, lane);
                }
            }
        }
        put(PREV, next);                                 // (chunk 0: rows that nobody reads)
        fetch(c - 2, next);
        __syncthreads();
        // ---- second half: gv
        const int lane = static_cast<int>(lane_now()), l16 = lane & 15, g = lane >> 4, to = tile_offset(l16, g, C);
        lds_t xo = sx + (16 * wz + l16) * A::ROW + 16 * g, ht = sb + A::DSH + (8 * g + (l16 >> 2)) * A::ROW + 8 * (l16 & 3) + 64 * wq;
        lds_t xt = sx + (4 * g + (l16 >> 2)) * A::ROW + 8 * (l16 & 3) + 64 * wq;
        opaque(xo); opaque(ht); opaque(xt);
        f32x4 O[2] = {ZERO4, ZERO4};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const Op2 ke = scaled(ld_op(xo + A::K + 64 * ks), cke[ks]);
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                const Op2 s = {ld_tr(ht + 32 * ks * A::ROW + 32 * ct, A::ROW), ld_tr(ht + (A::DSL - A::DSH) + 32 * ks * A::ROW + 32 * ct, A::ROW)};
                O[ct] = mm3(ke, s, O[ct]);
            }
        }
        const Op2 at = wz ? take_lane_tile<PARTS, A::PART, 1>(sb + A::BPART, lane) : take_lane_tile<PARTS, A::PART, 0>(sb + A::BPART, lane);
        const rows_t out = rows_of(p.gv + base + static_cast<size_t>(c) * L * C + 32 * wq, T - c * L, C);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const bf16x8 go = ld_tra<A::ROW>(xt + A::GY + 32 * ct);
            store_tile(out, to + 32 * wz * C + 32 * ct, C, l16, mfma(at.l, go, mfma(at.h, go, O[ct])));
        }
        tile_b(PREV);
        __syncthreads();
    };
    __syncthreads();
    tile_b(1);
    __syncthreads();
    for (int c = nch - 1; c >= 0; c -= 2) {
        chunk(std::true_type{}, c);
        chunk(std::false_type{}, c - 1);
    }
}

template <int HN>
__global__ __launch_bounds__(8 * HN, HN / 32) void wkv5b_bwd(const ArgsW p) {
    const lds_t sb = lds_of(smem_raw);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Part part = part_of(p, HN, true);              // (a last chunk without tokens adds zeros)
    if ((HN == 64 && !strong_layer(p.w, p.C, tid & 63)) || steps_head<false, HN>(p.w, nullptr, part.h * HN)) return;
    head_setup<HN>(p, sb, part, tid);
    __syncthreads();
    if (w < HN / 16) role_d<HN>(p, sb, w, tid & 63, part);
    else role_e<HN>(p, sb, tid - 4 * HN, part);
}

// gw, gu of a batch row from its blocks, rounded once
__global__ __launch_bounds__(256) void block_rows(int NB, size_t n, const float* __restrict__ w32, const float* __restrict__ u32, uint16_t* gw, uint16_t* gu) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const float* const x = (blockIdx.y == 0 ? w32 : u32) + i;
    float s = 0.f;
    for (int m = 0; m < NB; ++m) s += x[m * n];
    (blockIdx.y == 0 ? gw : gu)[i] = f2bf(s);
}

template <class F> int launch(F* kernel, hipStream_t st, const ArgsW& p, int threads, uint32_t lds) {
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)); e != hipSuccess) {
        g_last_hip_error = static_cast<int>(e);
        return RWKV_ERR_LAUNCH;
    }
    hipLaunchKernelGGL(kernel, dim3(p.heads * p.NB), dim3(threads), lds, st, p);
    return launch_status();
}

// Blocks of time, heads of 128 channels: as many as give every CU a workgroup (the kernels' LDS leaves room for one), of BLOCK_PAIRS pairs of
// chunks at least; 1: whole sequences.  per: pairs a block.  Where the line lies, B H sequences, us whole / in blocks: forward 8 of T400 34 / 30,
// of T4096 255 / 99; 64 of T400 34 / 34, of T4096 261 / 130; 128 of T400 36 / 43, of T800 60 / 61, of T2000 135 / 122; forward + backward 8 of
// T400 129 / 77, of T4096 1059 / 191; 32 of T4096 1095 / 251; 64 of T4096 1112 / 428; 128 of T400 136 / 116, of T4096 1153 / 821.
constexpr int BLOCK_PAIRS = 2, SLOTS = 256;
int time_blocks(int heads, int T, bool bwd, int* per) {
    const int want = SLOTS / heads;
    const int pairs = static_cast<int>((static_cast<long long>(T) + 2 * L - 1) / (2 * L));
    *per = pairs;
    if (want < 2 || pairs < 3 * BLOCK_PAIRS || (!bwd && pairs * 8 < heads)) return 1;
    const int least = static_cast<int>((pairs + want - 1) / want);
    *per = least > BLOCK_PAIRS ? least : BLOCK_PAIRS;
    return (pairs + *per - 1) / *per;
}
size_t round16(size_t x) { return (x + 15) & ~static_cast<size_t>(15); }
// Heads done as whole sequences, then others in NB blocks of `per` pairs.  The heads beyond a multiple of the CUs would be a last round of few
// workgroups, as long as the others.  us whole / split, forward, backward: 264 heads of T400 82 / 76, 202 / 157, of T2000 347 / 273, 814 / 539; 288 of T400
// 76 / 75, 200 / 163, of T2000 360 / 295, 833 / 588; 320 of T800 147 / 152, 357 / 283; 384 of T400 78 / ., 202 / 190, of T2000 390 / 387, 856 / 770; 528 of T800 230 /
// 218, 520 / 438; 576 of T800 243 / 272, 534 / 480.
struct SplitW { int whole, rest, NB, per; };
constexpr int REST_FWD = 32, REST_BWD = 128;
SplitW split_heads(int B, int T, int H, bool bwd) {
    if (static_cast<long long>(B) * H > 0x7fffffffLL) return {0, 0, 1, 0};      // (no memory holds them)
    const int all = B * H, rest = all % SLOTS;
    SplitW x{all - rest, rest, 1, 0};
    if (rest > 0 && (all < SLOTS || rest <= (bwd ? REST_BWD : REST_FWD))) x.NB = time_blocks(rest, T, bwd, &x.per);
    return x.NB > 1 ? x : SplitW{all, 0, 1, 0};
}
// whole sequences, then those in blocks (heads of 128): a launch each
template <bool REV, class F, class W> int in_parts(hipStream_t st, int B, ArgsW& p, void* ws, F* kernel, int threads, uint32_t lds, W after) {
    SplitW x = split_heads(B, p.T, p.H, REV);
    if (x.whole + x.rest == 0) return RWKV_ERR_SHAPE;
    if (ws == nullptr) x = {B * p.H, 0, 1, 0};
    p.heads = x.whole; p.at = 0; p.NB = 1; p.per = 0;
    if (x.whole > 0)
        if (int e = launch(kernel, st, p, threads, lds)) return e;
    if (x.rest == 0) return RWKV_OK;
    p.heads = x.rest; p.at = x.whole; p.NB = x.NB; p.per = x.per;
    p.local = static_cast<float*>(ws);
    p.gw32 = p.local + static_cast<size_t>(x.rest) * (x.NB - 1) * 128 * 128;
    p.gu32 = p.gw32 + static_cast<size_t>(x.NB) * x.rest * 128;
    hipLaunchKernelGGL((wkv5b_local<128, REV>), dim3(x.rest * (x.NB - 1)), dim3(256), 0, st, p);
    if (int e = launch(kernel, st, p, threads, lds)) return e;
    after();
    return launch_status();
}

}  // namespace

size_t wkv5b_saved_bytes(int B, int T, int C, int H) {
    const size_t nch = (static_cast<size_t>(T) + L - 1) / L, n = C / H;
    return static_cast<size_t>(B) * H * ((nch + 1) / 2) * n * n * sizeof(float);
}
size_t wkv5b_blocks_bytes(int B, int T, int C, int H, bool bwd) {
    if (C != H * 128) return 0;
    const SplitW x = split_heads(B, T, H, bwd);
    if (x.NB == 1) return 0;
    return static_cast<size_t>(x.rest) * (x.NB - 1) * 128 * 128 * sizeof(float) + (bwd ? round16(2 * static_cast<size_t>(x.NB) * x.rest * 128 * sizeof(float)) : 0);
}
int launch_wkv5b_fwd(hipStream_t st, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k, const uint16_t* v, const uint16_t* w,
                     const uint16_t* u, uint16_t* y, float* decay, float* saved, void* ws) {
    ArgsW p{};
    p.T = T; p.C = C; p.H = H; p.r = r; p.k = k; p.v = v; p.w = w; p.u = u; p.y = y; p.decay = decay; p.saved = saved;
    const auto none = []() {};
    if (C == H * 64) return in_parts<false>(st, B, p, nullptr, wkv5b_fwd<64>, NTH, G<64>::FTOTAL, none);
    return in_parts<false>(st, B, p, ws, wkv5b_fwd<128>, NTH, G<128>::FTOTAL, none);
}
int launch_wkv5b_bwd(hipStream_t st, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k, const uint16_t* v, const uint16_t* w,
                     const uint16_t* u, const uint16_t* gy, uint16_t* gr, uint16_t* gk, uint16_t* gv, uint16_t* gw, uint16_t* gu, const float* saved, void* ws) {
    ArgsW p{};
    p.T = T; p.C = C; p.H = H; p.r = r; p.k = k; p.v = v; p.w = w; p.u = u; p.gy = gy; p.gr = gr; p.gk = gk; p.gv = gv; p.gw = gw; p.gu = gu;
    p.saved = const_cast<float*>(saved);
    const auto rows = [&]() {
        const size_t n = static_cast<size_t>(p.heads) * 128, o = static_cast<size_t>(p.at) * 128;
        hipLaunchKernelGGL(block_rows, dim3(static_cast<unsigned>((n + 255) / 256), 2), dim3(256), 0, st, p.NB, n, p.gw32, p.gu32, gw + o, gu + o);
    };
    if (C == H * 64) return in_parts<true>(st, B, p, nullptr, wkv5b_bwd<64>, 512, G<64>::BTOTAL, rows);
    return in_parts<true>(st, B, p, ws, wkv5b_bwd<128>, 1024, G<128>::BTOTAL, rows);
}

}  // namespace rwkv
