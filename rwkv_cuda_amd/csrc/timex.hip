// depthwise_conv1d ("TimeX"): causal depthwise convolution with a full-length (T-tap) kernel
// per channel, fp32, gfx950.
//
//   x[b,c,t]  = eps + sum_{u<=t} wr[t-u] k[b,c,u]            wr[d] = w[c, T-1-d]
//   gk[b,c,u] =       sum_{t>=u} wr[t-u] g[b,c,t]
//   gw[b,c,T-1-d] =   sum_{u}    g[b,c,u+d] k[b,c,u]         (per batch; the wrapper sums over b)
//
// Two families on the matrix cores at fp32 accuracy: timex_conv_h2 / timex_gw_sum_h2 (two fp16 terms per operand) for whole tiles
// of 32 steps and full batches, timex_conv_any / timex_gw_any, timex_gw_short (three bf16 terms) for every other length and batch size.
// timex_gw (vector units) makes the per-batch gw of the reference's signature: one workgroup per (b,c) row; a thread owns 4
// consecutive lags d.
#include <algorithm>

#include "common.h"

namespace rwkv {
namespace {

// gw[row][T-1-d] = sum_u g[row][u+d] k[row][u]
__global__ __launch_bounds__(1024) void timex_gw(const float* __restrict__ k, const float* __restrict__ g,
                                                float* __restrict__ gw, int T) {
    extern __shared__ float lds[];
    float* ks = lds;                 // [T]
    float* gs = lds + T;             // [T + 4], four trailing zeros
    const size_t row = blockIdx.x;
    const int tid = threadIdx.x;
    *reinterpret_cast<float4*>(ks + 4 * tid) = *reinterpret_cast<const float4*>(k + row * T + 4 * tid);
    *reinterpret_cast<float4*>(gs + 4 * tid) = *reinterpret_cast<const float4*>(g + row * T + 4 * tid);
    for (int i = tid; i < 4; i += (T >> 2)) gs[T + i] = 0.f;
    __syncthreads();

    const int d0 = 4 * tid;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int u4 = 0; u4 + d0 < T; u4 += 4) {
        const float4 k4 = *reinterpret_cast<const float4*>(ks + u4);
        const float4 g0 = *reinterpret_cast<const float4*>(gs + u4 + d0);
        const float4 g1 = *reinterpret_cast<const float4*>(gs + u4 + d0 + 4);
        const float kv[4] = {k4.x, k4.y, k4.z, k4.w};
        const float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[a] = fmaf(gv[e + a], kv[e], acc[a]);   // g[u4+e + d0+a] k[u4+e]
    }
    // lags d0..d0+3 live at taps T-1-d0 .. T-4-d0
    *reinterpret_cast<float4*>(gw + row * T + (T - 4 - d0)) = make_float4(acc[3], acc[2], acc[1], acc[0]);
}

// ---------------------------------------------------------------------------------------------------- matrix-core path
// For T a multiple of 32 (and short enough for 32 rows to sit in LDS) the convolution of 32 batch rows of one channel is a
// product of the lower-triangular Toeplitz matrix W[t][u] = wr[t-u] with the [T x 32] block of inputs, on 32 x 32 matrix
// instructions (accumulator register v of lane l: row 8 (v/4) + 4 (l>>5) + (v&3), column l & 31).  The kernel row is
// followed by zeros, so a tap of negative lag reads 0 and the diagonal block needs no mask.  Output tile o of 32 time
// steps sums over input tiles 0..o (mirror: o..T/32-1); the tiles are dealt to the eight waves so that their loads are
// about equal.  256 persistent workgroups; a unit is one channel x 32 batch rows, and the next unit's rows are
// loaded into registers under the products of the current one.
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int MROWS = 32;              // batch rows per workgroup = columns of the product
constexpr int T_MFMA_MAX = 1024;
constexpr int TXW = 8;                 // waves per workgroup: two per SIMD, one reads LDS while the other runs MFMAs
constexpr int TXT = 64 * TXW;
constexpr int NCU = 256;               // workgroups of the persistent kernels: one per CU

// ------------------------------------------------------------------------------------ fp32 accuracy from fp16 x 2 products
// Every fp32 operand x is cut into two fp16 terms, x 2^s = h + l (h the nearest fp16, l the nearest fp16 of what h
// leaves: 22 mantissa bits together), and
//     x y = (h h' + h l' + l h') 2^-(s+s')                    (the term left out is below 2^-22 of the product)
// on v_mfma_f32_32x32x16_f16: three instructions of 16 matrix passes where v_mfma_f32_32x32x2_f32 needs eight of 16 passes
// for the same 32 x 32 x 16 block, i.e. 5.3 times the arithmetic rate at fp32 accuracy (accumulation is fp32 either way).
// fp16 has five exponent bits: the power of two 2^s brings the largest magnitude of a unit's rows (and of the kernel row)
// to [2^14, 2^15), computed for every unit from the rows themselves.  Elements more than 2^28 below that lose bits (fp16
// subnormals: absolute error 2^-25 on that scale, 2^-40 of the largest element), which a sum that contains the large
// elements does not see; the accumulators are scaled back exactly.
// Operand layout of the instruction: lane = (row or column l & 31, K half l >> 5) holds the eight consecutive K slots
// 8 (l >> 5) .. + 7; accumulator as above.  K slot s of a step is input step 16 ks + s of the 32-step tile.
//   rows : two planes [32 batch rows][T + 16] fp16; a lane's eight slots are 16 aligned bytes.
//   taps : the A operand of row t and slot u is line[base(t) + u] for a line that depends only on the direction
//          (forward: the kernel row in tap order followed by zeros; mirror: 31 zeros, then the reversed kernel row), so a
//          lane reads eight consecutive bf16 starting at an arbitrary element.  Two copies of every plane, the second
//          shifted by one element, make that four aligned dwords whatever the parity of the start.
// LDS: 2 x 32 x (T + 16) x 2 + 4 x (T + 96) x 2 + 64 bytes = 142 144 of 163 840 at T = 1024, the longest T this form takes.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
constexpr int T_H2_MAX = 1024;
constexpr int T_ANY = 4096;            // the longest sequence of the kernels for any shape
constexpr int T_H2_MID = 768;          // up to here a lane holds 3 pieces (16 bytes each) of each of its four rows while they are in flight, beyond 4
__host__ __device__ inline int h2_row_stride(int T) { return T + 16; }           // elements; (T + 16) / 2 dwords = 8 or 24 mod 32
__host__ __device__ inline int h2_line_len(int T) { return T + ((T & 32) ? 64 : 96); }    // half of it = 16 mod 32 dwords: the shifted copy sits 16 banks away
__host__ __device__ inline size_t h2_lds_bytes(int T) {
    return (2 * static_cast<size_t>(MROWS) * h2_row_stride(T) + 4 * static_cast<size_t>(h2_line_len(T))) * sizeof(uint16_t) + 16 * sizeof(float);
}
// x (already scaled) = h + l: h the nearest fp16, l the nearest fp16 of the exact remainder
struct H2 { uint16_t h, l; };
DEVINL H2 split2(float x) {
    const _Float16 h = static_cast<_Float16>(x);
    const _Float16 l = static_cast<_Float16>(x - static_cast<float>(h));
    H2 r;
    r.h = __builtin_bit_cast(uint16_t, h);
    r.l = __builtin_bit_cast(uint16_t, l);
    return r;
}
// the same for four elements times a power of two (the scaling is exact, so the remainder may be formed from x up in one
// fused operation): four multiplications, four fused multiply-adds and four packed conversions
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
struct H2x4 { uint2 h, l; };
DEVINL H2x4 split2x4(const float4& v, const float up) {
    const f32x2 a = {v.x * up, v.y * up}, b = {v.z * up, v.w * up};
    const f16x2 ha = __builtin_convertvector(a, f16x2), hb = __builtin_convertvector(b, f16x2);
    const f32x2 ra = a - __builtin_convertvector(ha, f32x2), rb = b - __builtin_convertvector(hb, f32x2);
    const f16x2 la = __builtin_convertvector(ra, f16x2), lb = __builtin_convertvector(rb, f16x2);
    H2x4 r;
    r.h = make_uint2(__builtin_bit_cast(uint32_t, ha), __builtin_bit_cast(uint32_t, hb));
    r.l = make_uint2(__builtin_bit_cast(uint32_t, la), __builtin_bit_cast(uint32_t, lb));
    return r;
}
// 2^s with m 2^s in [2^14, 2^15) for a magnitude m (s = 0 for zero, subnormal or infinite m), and 2^-s
struct Pow2 { float up, down; };
DEVINL Pow2 scale_for(float m) {
    const int e = static_cast<int>((__float_as_uint(m) >> 23) & 255u);
    int sft = 14 + 127 - e;
    sft = sft < -100 ? -100 : (sft > 100 ? 100 : sft);
    if (e == 0 || e == 255) sft = 0;
    Pow2 r;
    r.up = __uint_as_float(static_cast<uint32_t>(127 + sft) << 23);
    r.down = __uint_as_float(static_cast<uint32_t>(127 - sft) << 23);
    return r;
}
DEVINL float wave_max(float m) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    return m;
}
DEVINL float max_abs4(float m, const float4& v) { return fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w))); }

// NI: 16-byte pieces of a row per lane, 64 lanes a row: 3 up to T = 768, 4 beyond
template <bool MIRROR, int NI>
__global__ __launch_bounds__(TXT) void timex_conv_h2(const float* __restrict__ w, const float* __restrict__ in,
                                                      float* __restrict__ out, float eps, int B, int C, int T) {
    extern __shared__ float lds[];
    const int rs = h2_row_stride(T), xl = h2_line_len(T);
    uint16_t* rp = reinterpret_cast<uint16_t*>(lds);                    // [2][32][rs]
    uint16_t* al = rp + 2 * MROWS * rs;                                 // [2 planes][2 copies][xl]
    float* red = reinterpret_cast<float*>(al + 4 * xl);                 // [2][8]: every wave's largest magnitude of the rows / of the kernel row
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, kh = lane >> 5;
    const int q4n = T >> 2, nt = T >> 5;
    const int nbg = (B + MROWS - 1) / MROWS, nunits = C * nbg;
    // Staging: wave wv takes rows 4 wv .. 4 wv + 3 of the unit, lane l the 16-byte pieces l, l + 64, ... of each: a row's
    // address is wave-uniform, the rest is the lane number times 16 and a constant, in global memory and in LDS alike.
    float4 x[4][NI];
    float wr[2];
    // (in NI parts, piece i of the four rows each, the kernel row with part 0: asked for all at once by every workgroup of
    //  the chip at the same moment, the loads queue up in the memory system and the waves stall issuing them; the parts
    //  are spread over the products of the unit before)
    auto fetch_part = [&](const int unit, const int i) __attribute__((always_inline)) {
        const int c = unit / nbg, b0 = (unit - c * nbg) * MROWS;
        const int q4 = min(lane + 64 * i, q4n - 1);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            // (a row past the batch is read as the batch's last row and counts as zero later)
            const int b = min(b0 + 4 * wv + rr, B - 1);
            x[rr][i] = *reinterpret_cast<const float4*>(in + (static_cast<size_t>(b) * C + c) * T + 4 * q4);
        }
        if (i == 0) {
#pragma unroll
            for (int s = 0; s < 2; ++s) wr[s] = w[static_cast<size_t>(c) * T + min(s * TXT + tid, T - 1)];
        }
    };
    // the largest magnitudes of the unit, this wave's part (pieces past a row's end repeat its last piece)
    auto unit_max = [&]() __attribute__((always_inline)) {
        float mx = 0.f;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
#pragma unroll
            for (int i = 0; i < NI; ++i) mx = max_abs4(mx, x[rr][i]);
        mx = wave_max(mx);
        const float mw = wave_max(fmaxf(fabsf(wr[0]), fabsf(wr[1])));
        if (lane == 0) { red[wv] = mx; red[8 + wv] = mw; }
    };
    float unscale = 1.f;
    auto store_unit = [&](const int unit) __attribute__((always_inline)) {
        const int c = unit / nbg, b0 = (unit - c * nbg) * MROWS;
        float mx = 0.f, mw = 0.f;
#pragma unroll
        for (int i = 0; i < TXW; ++i) { mx = fmaxf(mx, red[i]); mw = fmaxf(mw, red[8 + i]); }
        const Pow2 sx = scale_for(mx), sw = scale_for(mw);
        unscale = sx.down * sw.down;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const int r = 4 * wv + rr;
            const float up = b0 + r < B ? sx.up : 0.f;
            uint16_t* d = rp + r * rs + 4 * lane;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if (lane + 64 * i < q4n) {
                    const H2x4 y = split2x4(x[rr][i], up);
                    *reinterpret_cast<uint2*>(d + 256 * i) = y.h;
                    *reinterpret_cast<uint2*>(d + 256 * i + MROWS * rs) = y.l;
                }
            }
        }
        // tap tau of the kernel row sits at line position tau (forward) or 31 + (T - 1 - tau) (mirror); the rest is zero
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int tau = s * TXT + tid;
            if (tau < T) {
                const H2 a = split2(wr[s] * sw.up);
                const int pos = MIRROR ? 31 + (T - 1 - tau) : tau;
                const uint16_t pl[2] = {a.h, a.l};
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    al[(2 * p) * xl + pos] = pl[p];
                    if (pos >= 1) al[(2 * p + 1) * xl + pos - 1] = pl[p];
                }
            }
        }
        (void)c;
    };
    // the zero parts of the line never change: clear everything once (the taps are rewritten for every unit)
    for (int i = tid; i < 4 * xl; i += TXT) al[i] = 0;
    __syncthreads();
    int unit = blockIdx.x;
    if (unit < nunits) {
#pragma unroll
        for (int i = 0; i < NI; ++i) fetch_part(unit, i);
    }
    static_assert(T_H2_MAX / 64 <= 2 * TXW, "a wave takes at most two pairs of tiles per unit");

    for (; unit < nunits; unit += gridDim.x) {
        const int c = unit / nbg, b0 = (unit - c * nbg) * MROWS;
        unit_max();
        __syncthreads();
        store_unit(unit);
        __syncthreads();
        const int next = unit + static_cast<int>(gridDim.x);
        const bool more = next < nunits;
        if (more) fetch_part(next, 0);
        // Output tile ot sums over ot + 1 input tiles (mirror: T/32 - ot).  A wave works on two neighbouring output tiles at a
        // time, because they share operands: a step is 16 input steps (K = 16), and with
        //   forward: row t = 32 ot + ln, slot u: tap T-1-(t-u)            -> line[T-1-32 ot-ln + u],  rows[u]
        //   mirror : row u = 32 ot + ln, slot t: lag 32 (it-ot) + slot-ln -> line[31-ln + 32 (it-ot) + slot],  rows[32 ot + slot]
        // step j of both tiles takes the same rows (forward) or the same taps (mirror), and the other operand of the
        // shorter tile at step j is that of the longer one (forward: tile ot + 1, mirror: tile ot) at step j + 2.  So a
        // step reads one operand of each kind from LDS (4 KB per wave) for six matrix instructions instead of three: the
        // "carried" operand C(j) enters the shorter tile at once and the longer tile two steps later, from registers.
        // The pairs are dealt to the waves in the order of decreasing work, back and forth (waves 0..7, then 7..0): at most
        // two pairs a wave.
        const int npairs = (nt + 1) >> 1;
        auto do_pair = [&](const int ts, auto&& halfway) __attribute__((always_inline)) {
            {
                const int m = MIRROR ? ts : npairs - 1 - ts;
                // the longer tile and the shorter one (absent when T/32 is odd and this is the last tile)
                const bool both = 2 * m + 1 < nt;
                const int tl = MIRROR ? 2 * m : (both ? 2 * m + 1 : 2 * m), tsh = MIRROR ? 2 * m + 1 : 2 * m;
                const int n_long = 2 * (MIRROR ? nt - tl : tl + 1), n_short = n_long - 2;
                f32x16 accl, accs;                             // the two tiles' instructions alternate: consecutive ones are independent
#pragma unroll
                for (int v = 0; v < 16; ++v) { accl[v] = 0.f; accs[v] = 0.f; }
                const int start0 = (MIRROR ? 31 - ln : T - 1 - 32 * tl - ln) + 8 * kh;
                const uint32_t* ap0 = reinterpret_cast<const uint32_t*>(al + (start0 & 1) * xl) + (start0 >> 1);
                const uint16_t* bp0 = rp + ln * rs + (MIRROR ? 32 * tl : 0) + 8 * kh;
                auto taps = [&](int j, f16x8 (&f)[2]) __attribute__((always_inline)) {
#pragma unroll
                    for (int pq = 0; pq < 2; ++pq) {
                        const uint32_t* a4 = ap0 + 8 * j + pq * xl;    // a plane is 2 xl elements = xl dwords
                        f[pq] = __builtin_bit_cast(f16x8, make_uint4(a4[0], a4[1], a4[2], a4[3]));
                    }
                };
                auto rows = [&](int j, f16x8 (&f)[2]) __attribute__((always_inline)) {
#pragma unroll
                    for (int pq = 0; pq < 2; ++pq) f[pq] = __builtin_bit_cast(f16x8, *reinterpret_cast<const uint4*>(bp0 + 16 * j + pq * MROWS * rs));
                };
                auto carried = [&](int j, f16x8 (&f)[2]) __attribute__((always_inline)) { if constexpr (MIRROR) rows(j, f); else taps(j, f); };
                auto shared = [&](int j, f16x8 (&f)[2]) __attribute__((always_inline)) { if constexpr (MIRROR) taps(j, f); else rows(j, f); };
                // term number `term` of the product of a carried and a shared operand: h h', h l', l h'
                auto product = [&](f32x16& acc, const int term, const f16x8 (&cc)[2], const f16x8 (&sh)[2]) __attribute__((always_inline)) {
                    const f16x8 (&fa)[2] = MIRROR ? sh : cc;
                    const f16x8 (&fb)[2] = MIRROR ? cc : sh;
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[term == 2 ? 1 : 0], fb[term == 1 ? 1 : 0], acc, 0, 0, 0);
                };
                // (a last tile without a partner computes a second tile all the same and does not store it)
                auto step = [&](const f16x8 (&cl)[2], const f16x8 (&cs)[2], const f16x8 (&sh)[2]) __attribute__((always_inline)) {
#pragma unroll
                    for (int term = 0; term < 3; ++term) { product(accl, term, cl, sh); product(accs, term, cs, sh); }
                };
                // Two pairs of carried operands, P and Q, change roles every two steps (the longer tile reads what the shorter
                // one read two steps earlier), the shared operand alternates between two sets: no register is ever copied.
                // Every read is issued one step ahead; the fences keep it in front of the products of the current step.
                // (C(j) is asked for up to j = n_long - 1 only, S(j) likewise: nothing outside the tiles' own steps is read.)
                f16x8 P[2][2], Q[2][2], se[2], so[2];
                carried(0, P[0]); carried(1, P[1]); carried(n_long > 2 ? 2 : 1, Q[0]); shared(0, se);
                // (one way into every loop body and one way out: with an exit in the middle of a body the compiler keeps two
                //  versions of the accumulators and copies all 32 registers between them in every pass of the loop, after waiting for
                //  the matrix pipeline to drain)
                auto block_pq = [&](const int j) __attribute__((always_inline)) {      // steps j, j + 1: longer tile from P, shorter from Q
                    carried(j + 3, Q[1]); shared(j + 1, so);
                    __builtin_amdgcn_sched_barrier(0);
                    step(P[0], Q[0], se);
                    __builtin_amdgcn_sched_barrier(0);
                    carried(min(j + 4, n_long - 1), P[0]); shared(j + 2, se);
                    __builtin_amdgcn_sched_barrier(0);
                    step(P[1], Q[1], so);
                    __builtin_amdgcn_sched_barrier(0);
                };
                auto block_qp = [&](const int j) __attribute__((always_inline)) {      // the same with the roles of P and Q exchanged
                    carried(j + 3, P[1]); shared(j + 1, so);
                    __builtin_amdgcn_sched_barrier(0);
                    step(Q[0], P[0], se);
                    __builtin_amdgcn_sched_barrier(0);
                    carried(min(j + 4, n_long - 1), Q[0]); shared(j + 2, se);
                    __builtin_amdgcn_sched_barrier(0);
                    step(Q[1], P[1], so);
                    __builtin_amdgcn_sched_barrier(0);
                };
                int j = 0;
                const int half = (n_short >> 1) & ~3;
                for (; j < half; j += 4) { block_pq(j); block_qp(j + 2); }
                halfway();
                for (; j + 4 <= n_short; j += 4) { block_pq(j); block_qp(j + 2); }
                if (j < n_short) {                              // (two steps left: afterwards the longer tile's operands are in Q)
                    block_pq(j);
#pragma unroll
                    for (int q = 0; q < 2; ++q) { P[0][q] = Q[0][q]; P[1][q] = Q[1][q]; }
                }
                // the last two steps belong to the longer tile alone
                shared(n_short + 1, so);
#pragma unroll
                for (int term = 0; term < 3; ++term) product(accl, term, P[0], se);
#pragma unroll
                for (int term = 0; term < 3; ++term) product(accl, term, P[1], so);
                auto put_tile = [&](f32x16& acc, const int ot) __attribute__((always_inline)) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[v] = fmaf(acc[v], unscale, MIRROR ? 0.f : eps);
                    if (b0 + ln < B) {
                        float* o = out + (static_cast<size_t>(b0 + ln) * C + c) * T + 32 * ot + 4 * kh;
#pragma unroll
                        for (int v4 = 0; v4 < 4; ++v4)
                            *reinterpret_cast<float4*>(o + 8 * v4) = make_float4(acc[4 * v4], acc[4 * v4 + 1], acc[4 * v4 + 2], acc[4 * v4 + 3]);
                    }
                };
                put_tile(accl, tl);
                if (both) put_tile(accs, tsh);
            }
        };
        if (wv < npairs) do_pair(wv, [&]() __attribute__((always_inline)) { if (more) fetch_part(next, 1); });
        else if (more) fetch_part(next, 1);
        if (more) fetch_part(next, 2);
        if (2 * TXW - 1 - wv < npairs) do_pair(2 * TXW - 1 - wv, []() __attribute__((always_inline)) {});
        if constexpr (NI > 3) { if (more) fetch_part(next, 3); }
        __syncthreads();               // every wave is done with this unit's rows
    }
}

// Kernel gradient summed over the batch: gws[c][T-1-lag] = sum_b sum_t g[b,c,t] k[b,c,t-lag], i.e. the sum of the lag-th
// sub-diagonal of M = G^T K (contraction over the batch), with the two-term fp16 products of timex_conv_h2.  Batch rows
// are staged 16 at a time (a pass; both tensors scaled by a power of two of their own per pass): one
// v_mfma_f32_32x32x16_f16 block per pair of tiles and product, K = the 16 batch rows.  A wave owns whole lag tiles d (all
// tile pairs (d + i, i) accumulate into the same registers); no atomics, every fp32 sum in a fixed order.
// The planes keep the tensors' own layout, [16 rows][T + 16 .. 112] fp16 (staged like the convolution's rows: a wave takes two
// rows of each tensor, wave-uniform row addresses, 8-byte LDS stores).  Both operands need the batch rows along K and a
// lane per step: ds_read_b64_tr_b16 delivers exactly that -- within 16 lanes, four rows of 16 consecutive steps come back
// with a lane per step and the four rows in its registers; two such reads are a lane's eight K slots.
// Two neighbouring lag tiles per wave at a time: tile pair i of lag tile d + 1 takes the same k tile as pair i of lag
// tile d, and its g tile is the one that lag tile d takes at pair i + 1.  So a pair reads one g tile and one k tile
// from LDS for six matrix instructions; the g operand enters lag tile d + 1 at once and lag tile d one pair later.
// A finished tile's diagonals are summed in registers: lane p of a half-wave collects, for every row t it holds, the
// element of column (t - p) mod 32 (one ds_bpermute per accumulator register), which belongs to diagonal p if t >= p and
// to diagonal p - 32 otherwise.
// LDS: 2 x 2 x 16 x (T + 16) x 2 + 2 T x 4 + 64 bytes = 141 376 at T = 1024.
constexpr int GH2_ROWS = 16;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef v4s __attribute__((address_space(3))) * lds_v4s_ptr;
// elements; = 16 mod 128, i.e. 8 banks mod 64: the 16 lanes of a transposing read take four rows x four 8-byte pieces, and
// with rows 8 banks apart the sixteen pieces fall on different banks
__host__ __device__ inline int gw_row_stride(int T) { return T + ((144 - (T & 127)) & 127); }
__host__ __device__ inline size_t gw_h2_lds_bytes(int T) {
    return 4 * static_cast<size_t>(GH2_ROWS) * gw_row_stride(T) * sizeof(uint16_t) + (2 * static_cast<size_t>(T) + 16) * sizeof(float);
}

// NI: 16-byte pieces of a row per lane, 64 lanes a row: 3 up to T = 768, 4 beyond
template <int NI>
__global__ __launch_bounds__(TXT) void timex_gw_sum_h2(const float* __restrict__ k, const float* __restrict__ g,
                                                        float* __restrict__ gws, int B, int C, int T) {
    extern __shared__ float lds[];
    const int rsg = gw_row_stride(T);
    const int plane = GH2_ROWS * rsg;                          // elements
    uint16_t* gp = reinterpret_cast<uint16_t*>(lds);           // [2][16][rsg]
    uint16_t* kp = gp + 2 * plane;                             // [2][16][rsg]
    float* diag = reinterpret_cast<float*>(kp + 2 * plane);    // [T/32 lag tiles][64]: entry l of tile d is the sum for lag 32 d + l - 31
    float* red = diag + 2 * T;                                 // [2][8]: every wave's largest magnitude of g / of k in this pass
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, kh = lane >> 5, l16 = lane & 15;
    const int nt = T >> 5, q4n = T >> 2;
    const int npass = (B + GH2_ROWS - 1) / GH2_ROWS;
    const int nmine = (C > static_cast<int>(blockIdx.x) ? (C - 1 - static_cast<int>(blockIdx.x)) / static_cast<int>(gridDim.x) + 1 : 0) * npass;
    // Staging: wave wv takes rows 2 wv and 2 wv + 1 of the pass, of both tensors; lane l the 16-byte pieces l, l + 64, ...
    float4 xg[2][NI], xk[2][NI];
    // (in NI parts, piece i of both rows and both tensors each: asked for all at once by every workgroup of the chip at the
    //  same moment, the loads queue up in the memory system and the waves stall issuing them while the matrix cores wait;
    //  the parts are spread over the products of the pass before)
    const int nblk = gridDim.x;
    auto fetch_part = [&](const int u, const int i) __attribute__((always_inline)) {
        const int c = blockIdx.x + (u / npass) * nblk, b0 = (u % npass) * GH2_ROWS;
        const int q4 = min(lane + 64 * i, q4n - 1);
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            // (a row past the batch is read as the batch's last row and counts as zero later)
            const size_t row = (static_cast<size_t>(min(b0 + 2 * wv + rr, B - 1)) * C + c) * T;
            xg[rr][i] = *reinterpret_cast<const float4*>(g + row + 4 * q4);
            xk[rr][i] = *reinterpret_cast<const float4*>(k + row + 4 * q4);
        }
    };
    // the largest magnitudes of the pass, this wave's part (pieces past a row's end repeat its last piece)
    auto unit_max = [&]() __attribute__((always_inline)) {
        float mg = 0.f, mk = 0.f;
#pragma unroll
        for (int rr = 0; rr < 2; ++rr)
#pragma unroll
            for (int i = 0; i < NI; ++i) { mg = max_abs4(mg, xg[rr][i]); mk = max_abs4(mk, xk[rr][i]); }
        mg = wave_max(mg); mk = wave_max(mk);
        if (lane == 0) { red[wv] = mg; red[8 + wv] = mk; }
    };
    float unscale = 1.f;
    auto store_unit = [&](const int u) __attribute__((always_inline)) {
        const int b0 = (u % npass) * GH2_ROWS;
        float mg = 0.f, mk = 0.f;
#pragma unroll
        for (int i = 0; i < TXW; ++i) { mg = fmaxf(mg, red[i]); mk = fmaxf(mk, red[8 + i]); }
        const Pow2 sg = scale_for(mg), sk = scale_for(mk);
        unscale = sg.down * sk.down;
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            const int r = 2 * wv + rr;
            const bool real = b0 + r < B;
            const float ug = real ? sg.up : 0.f, uk = real ? sk.up : 0.f;
            uint16_t* dg = gp + r * rsg + 4 * lane;
            uint16_t* dk = kp + r * rsg + 4 * lane;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if (lane + 64 * i < q4n) {
                    const H2x4 yg = split2x4(xg[rr][i], ug), yk = split2x4(xk[rr][i], uk);
                    *reinterpret_cast<uint2*>(dg + 256 * i) = yg.h;
                    *reinterpret_cast<uint2*>(dg + 256 * i + plane) = yg.l;
                    *reinterpret_cast<uint2*>(dk + 256 * i) = yk.h;
                    *reinterpret_cast<uint2*>(dk + 256 * i + plane) = yk.l;
                }
            }
        }
    };
    // operand of tile tt of a tensor: lane (ln, kh) <-> step 32 tt + ln, K slot 8 kh + e <-> batch row 8 kh + e.  Within its
    // group of 16 lanes a lane points at [row 8 kh + (l16 >> 2)][step 32 tt + 16 (ln >> 4) + 4 (l16 & 3)]; the second read
    // is four rows further on.
    const uint32_t tr0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)gp))
                       + 2u * static_cast<uint32_t>((8 * kh + (l16 >> 2)) * rsg + 16 * (ln >> 4) + 4 * (l16 & 3));
    const uint32_t k_off = 2u * 2u * static_cast<uint32_t>(plane), row4 = 2u * 4u * static_cast<uint32_t>(rsg), pl_b = 2u * static_cast<uint32_t>(plane);
    auto operand = [&](const uint32_t base, const int tt, f16x8 (&f)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int pq = 0; pq < 2; ++pq) {
            const uint32_t a = base + 64u * static_cast<uint32_t>(tt) + pq * pl_b;
            const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(a));
            const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(a + row4));
            const uint2 x = __builtin_bit_cast(uint2, lo), y = __builtin_bit_cast(uint2, hi);
            f[pq] = __builtin_bit_cast(f16x8, make_uint4(x.x, x.y, y.x, y.y));
        }
    };
    if (nmine > 0) {
#pragma unroll
        for (int i = 0; i < NI; ++i) fetch_part(0, i);
    }
    static_assert(T_H2_MAX / 64 <= 2 * TXW, "a wave takes at most two pairs of lag tiles per pass");

    for (int u = 0; u < nmine; ++u) {
        const int pass = u % npass;
        if (pass == 0)
            for (int i = tid; i < 2 * T; i += TXT) diag[i] = 0.f;
        unit_max();
        __syncthreads();
        store_unit(u);
        __syncthreads();
        const bool more = u + 1 < nmine;
        if (more) fetch_part(u + 1, 0);
        // lag tile d has T/32 - d tile pairs; the lag tiles go to the waves two at a time (2 m, 2 m + 1), in the order of
        // decreasing work, back and forth (waves 0..7, then 7..0): at most two pairs a wave
        const int npairs = (nt + 1) >> 1;
        auto do_pair = [&](const int m, auto&& halfway) __attribute__((always_inline)) {
            const int dl = 2 * m, n = nt - dl;                 // the longer lag tile and its tile pairs; the shorter one, dl + 1, has n - 1
            f32x16 accl, accs;
#pragma unroll
            for (int v = 0; v < 16; ++v) { accl[v] = 0.f; accs[v] = 0.f; }
            // term number `term` of the product of a g and a k operand: h h', h l', l h'
            auto product = [&](f32x16& acc, const int term, const f16x8 (&fa)[2], const f16x8 (&fb)[2]) __attribute__((always_inline)) {
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[term == 2 ? 1 : 0], fb[term == 1 ? 1 : 0], acc, 0, 0, 0);
            };
            auto both = [&](const f16x8 (&al_)[2], const f16x8 (&as_)[2], const f16x8 (&fb)[2]) __attribute__((always_inline)) {
                // (the longer tile's first two terms go first: the shorter tile's g operand is the read issued last)
                product(accl, 0, al_, fb); product(accl, 1, al_, fb);
                product(accs, 0, as_, fb); product(accl, 2, al_, fb);
                product(accs, 1, as_, fb); product(accs, 2, as_, fb);
            };
            auto last = [&](const f16x8 (&al_)[2], const f16x8 (&fb)[2]) __attribute__((always_inline)) {
#pragma unroll
                for (int term = 0; term < 3; ++term) product(accl, term, al_, fb);
            };
            // Pair i: the longer lag tile takes g tile dl + i, the shorter one g tile dl + 1 + i, both k tile i.  Two sets of g
            // operands change roles every pair, two sets of k operands alternate; a set is read again as soon as its last
            // product has been issued, one pair ahead of its use.
            f16x8 P[2], Q[2], be[2], bo[2];
            operand(tr0, dl, P); operand(tr0 + k_off, 0, be); operand(tr0, min(dl + 1, nt - 1), Q);
            // (one way into the loop body and one way out, see timex_conv_h2)
            auto two_pairs = [&](const int i) __attribute__((always_inline)) {
                operand(tr0 + k_off, i + 1, bo);
                __builtin_amdgcn_sched_barrier(0);
                both(P, Q, be);
                __builtin_amdgcn_sched_barrier(0);
                operand(tr0, min(dl + 2 + i, nt - 1), P);
                operand(tr0 + k_off, i + 2, be);
                __builtin_amdgcn_sched_barrier(0);
                both(Q, P, bo);
                __builtin_amdgcn_sched_barrier(0);
                operand(tr0, min(dl + 3 + i, nt - 1), Q);
            };
            int i = 0;
            const int half = ((n - 1) >> 1) & ~1;
            for (; i < half; i += 2) two_pairs(i);
            halfway();
            for (; i + 2 <= n - 1; i += 2) two_pairs(i);
            if (i < n - 1) {                                    // one pair with both tiles left, then the longer tile's last pair
                operand(tr0 + k_off, i + 1, bo);
                __builtin_amdgcn_sched_barrier(0);
                both(P, Q, be);
                __builtin_amdgcn_sched_barrier(0);
                last(Q, bo);
            } else last(P, be);
            // accumulator v: t = 8 (v/4) + 4 kh + (v&3), u = ln, of tiles d apart
            auto diagonals = [&](const f32x16& acc, const int d) __attribute__((always_inline)) {
                float pos = 0.f, neg = 0.f;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int t = 8 * (v >> 2) + 4 * kh + (v & 3);
                    const float y = __shfl(acc[v], (kh << 5) | ((t - ln) & 31), 64);
                    if (t >= ln) pos += y; else neg += y;
                }
                pos += __shfl_xor(pos, 32, 64);
                neg += __shfl_xor(neg, 32, 64);
                if (kh == 0) diag[64 * d + 31 + ln] += pos * unscale;    // lag tile d belongs to this wave alone
                else if (ln >= 1) diag[64 * d + ln - 1] += neg * unscale;
            };
            diagonals(accl, dl);
            if (dl + 1 < nt) diagonals(accs, dl + 1);
        };
        if (wv < npairs) do_pair(wv, [&]() __attribute__((always_inline)) { if (more) fetch_part(u + 1, 1); });
        else if (more) fetch_part(u + 1, 1);
        if (more) fetch_part(u + 1, 2);
        if (2 * TXW - 1 - wv < npairs) do_pair(2 * TXW - 1 - wv, []() __attribute__((always_inline)) {});
        if constexpr (NI > 3) { if (more) fetch_part(u + 1, 3); }
        __syncthreads();
        if (pass == npass - 1) {
            const int c = blockIdx.x + (u / npass) * gridDim.x;
            for (int x = tid; x < T; x += TXT) {        // lag = 32 d + e comes from tile d (diagonal e) and tile d + 1 (diagonal e - 32)
                const int lag = T - 1 - x, d = lag >> 5, e = lag & 31;
                gws[static_cast<size_t>(c) * T + x] = diag[64 * d + 31 + e] + (d + 1 < nt ? diag[64 * (d + 1) + e - 1] : 0.f);
            }
            __syncthreads();           // diag is cleared for the next channel only after it has been read
        }
    }
}

// ------------------------------------------------------------------------------------ any length, any batch size
// The same products with the columns taken from time as well as from the batch.  With t = 32 a + i the convolution of a row is
//     out[32 a + i] = sum_{d <= a} sum_j W_d[i][j] in[32 (a - d) + j],     W_d[i][j] = wr[32 d + i - j],
// so for every block lag d one 32 x 32 Toeplitz matrix meets ALL 32-step blocks of all rows: a column is a pair (block a, row
// b), numbered a Bg + b in a unit of Bg batch rows of one channel, and 32 consecutive columns are a tile of one matrix
// instruction.  Two rows of 1500 steps fill three column tiles, where a tile of 32 batch rows would be empty but for two.
// A tile's columns differ in a by at most 31 / Bg: d runs to the largest a, and blocks before a row's start (mirror: after its
// end) read as zeros, of which every row has zb behind it.  The kernel gradient takes 256 lags a tile, d = i' + 8 j + 128 h with (i', h) the
// rows and j the columns of one 16 x 16 instruction, and time as its contraction:
//     M[(i', h)][j] = sum_t g[t + i' + 128 h] k[t - 8 j],
// a Hankel operand (the windows of g) and one whose columns begin 8 steps apart, so that every element is a tap: nothing is summed over
// diagonals, and the sums of all rows that a workgroup does stay in registers.  (Lag tiles of 32, columns (block, row) as above, whose
// sub-diagonals are summed after every few instructions, are timex_gw_short.)
// Which of the two a shape takes: gw_plan.
// Operands are THREE bf16 terms, x = h + m + l (each the nearest of what is left: all 24 bits of x), and a product is
//     x y = h h' + h m' + m h' + m m' + h l' + l h'            (the terms left out are below 2^-24 of the product, 2^-26 rms)
// with fp32's exponents.  The five small products have accumulators of their own: the sum of the large ones, whose roundings are
// what is left of an error, rounds once an instruction.  Nothing is scaled, so an element's accuracy does not depend on its
// neighbours: short rows, rows that grow late and batches of unequal rows come out as from an fp32 loop, which two fp16 terms
// under a common power of two (half the products, 58 and 101 us where these took 95 and 111) do not give.  A unit with an element that is no number, infinite or beyond
// bf16's largest is done by such a loop (a matrix product would carry it to earlier steps: zero times infinity).
// Rows lie in LDS as blocks of 32 + 8 terms (80 bytes: 16-byte reads of neighbouring columns fall on different banks if a
// row has an odd number of blocks), 512 threads, 128 registers, and at most 80 KB: two
// workgroups share a CU, one converts its rows while the other multiplies.  B13 C384 T1500:
// 77 us a convolution (92 with a wave per column tile and units of 4, 4, 4 and 1 rows; matrix pipes busy 70 % of the time that a CU has
// work), 77 us the kernel gradient (107 as lag tiles of 32), relative errors 1.8e-7 and 1.0e-7; the fp32 loops on the vector units
// that these replace took 315 / 286 and, with the sum over the batch, 243 us, with 5.6e-7.
constexpr int BLK = 40;                // elements of a block in LDS, 32 of them data
constexpr int LDS_CU = 160 * 1024, LDS_ANY = LDS_CU / 2;     // two workgroups per CU
constexpr int PZ = 32;                 // zeros in front of the forward line (lags beyond the last tap, of rows past T)
constexpr int CONV_PIECES = 8, GW_PIECES = 3;   // 16-byte pieces a thread stages (per tensor): Bg nt 8 / 512 at most
constexpr int NPL = 3;                 // planes: terms of an operand
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// the six products of two operands, the small ones first
constexpr int TERM_A[6] = {2, 0, 1, 1, 0, 0}, TERM_B[6] = {0, 2, 1, 0, 1, 0};

// Division by sizes of a launch, a multiplication and a shift: a real one is 30 vector instructions in kernels whose waves issue some 800.
// Exact for a column (at most 512) over rows (at most 32) and a zero block's number (at most 32 33) over the zero blocks of a row (at most 32):
// x (d - 1) < 2^16; and for a piece (at most 512) over the pieces of a row (at most 1024).
__host__ __device__ inline uint32_t inv16(int d) { return (65536u + d - 1) / d; }
__host__ __device__ inline uint32_t inv_per(int d) { return ((1u << 20) + d - 1) / d; }
__host__ __device__ inline int over16(int x, uint32_t inv) { return static_cast<int>(static_cast<uint32_t>(x) * inv >> 16); }
__host__ __device__ inline int over_per(int x, uint32_t inv) { return static_cast<int>(static_cast<uint32_t>(x) * inv >> 20); }
struct AnyGeom {
    int nt, bg, zb, pitch;             // blocks of a row, rows of a unit, zero blocks behind a row, nt + zb (odd)
    uint32_t bg_inv, zb_inv, per_inv;
    __host__ __device__ size_t plane() const { return static_cast<size_t>(zb + bg * pitch) * BLK; }     // elements
};
inline AnyGeom any_geom(int T, int bg, int span) {        // span: how many blocks the columns of one operand may differ by
    AnyGeom q;
    q.nt = (T + 31) / 32; q.bg = bg;
    q.zb = (span + bg - 1) / bg;
    q.zb += (q.nt + q.zb + 1) & 1;
    q.pitch = q.nt + q.zb;
    q.bg_inv = inv16(bg); q.zb_inv = inv16(q.zb); q.per_inv = inv_per(8 * q.nt);
    return q;
}
// What the eight waves of a workgroup of timex_conv_any do.  A pair of column tiles, neighbours in the order of decreasing work, needs
// its longer tile's block lags once for both (they share the Toeplitz operand); its lags are cut into runs of about equal work, a
// wave each, as many as it takes for the eight waves to be done at about the same time.  Wave w: lags d0 .. d1 - 1 of pair `pair`
// (NO_PAIR: nothing to do).  The pair's lowest wave adds the others' sums to its own and stores the tiles.
// (A tile of 1500 steps has up to 47 lags and there are six tiles of four rows: one wave a tile, or two short tiles, left two waves without
// work and the others waiting for the one with 47: B13 C384 T1500 92 us a convolution, 77 so.)
constexpr int NO_PAIR = 255;
struct ConvPlan {
    AnyGeom q;
    int shared;                        // whether a pair has more than one wave
    uint64_t pair, d0, d1;             // a byte a wave: read once, where bytes read one by one are a trip to memory each
    __host__ __device__ static int of(uint64_t x, int w) { return static_cast<int>(x >> (8 * w) & 255); }
};
static_assert(TXW == 8, "a word holds a byte a wave");
static_assert(T_ANY / 32 < 255, "a block lag is a byte");
// copies: of the taps' line.  With the second one, shifted by one, an odd window begins at a whole dword as an even one does; with one it is
// five dwords, shifted in registers, which makes room for a second workgroup on a CU beyond T = 3360: B1 C1024 T4096 forward + backward 297 us
// with two copies, 265 with one; T1500 with two 212, with one 216.
struct ConvPlans { ConvPlan p[2]; int copies, pairs; };   // p: for units of ceil(B / groups) and of floor(B / groups) rows; pairs: which kernel
__host__ __device__ inline int tile_lags(const AnyGeom& q, bool mirror, int tile) {
    const int ncol = q.nt * q.bg, last = 32 * tile + 31 < ncol ? 32 * tile + 31 : ncol - 1;
    return mirror ? q.nt - over16(32 * tile, q.bg_inv) : over16(last, q.bg_inv) + 1;
}
// tile number `rank` in the order of decreasing work; none: -1
__host__ __device__ inline int tile_of(int ntile, bool mirror, int rank) { return rank < ntile ? (mirror ? rank : ntile - 1 - rank) : -1; }
constexpr size_t SUM_SLOT = 2 * 32 * 32;      // floats of a wave's two tiles
inline size_t conv_any_lds(const AnyGeom& q, int copies) { return (NPL * q.plane() + copies * NPL * static_cast<size_t>(h2_line_len(32 * q.nt))) * 2 + 16; }

// The kernel gradient.  In LDS g lies in blocks of 128 steps and the GW_OVER - 128 after them (a window of eight steps is read within one
// block), a zero block behind, which is also what lies in front of k.  A window that begins at an odd step is the same five dwords as
// the one before it, shifted in registers (a second copy of g, shifted by one step, is half as many rows in LDS and four more writes a
// piece and term: B32 C1000 T36 18.9 us, 16.2 so).  A read of half a wave takes eight or nine dwords each from two blocks in a row, which are 8 banks
// apart (at the same bank such reads took twice as long, and they were as many cycles of LDS as those of k).
constexpr int GW_OVER = 144;
constexpr int GW_TILES = 8;            // lag tiles of a wave, 256 lags each
constexpr int GW_WAVES = 6;            // of more than eight tiles (T > 2048): the waves that take the first eight, which have about three times the work
struct GwGeom {
    int nt, bg, k, plane;              // elements from a plane's start to k, to the next plane
    uint32_t per_inv;
    __host__ __device__ int bytes() const { return bg * NPL * plane * 2 + 16; }
};
inline GwGeom gw_geom(int T, int bg) {
    GwGeom q;
    q.nt = (T + 31) / 32; q.bg = bg;
    q.k = GW_OVER * ((q.nt + 3) / 4 + 1);
    q.plane = q.k + 32 * q.nt;
    q.per_inv = inv_per(8 * q.nt);
    return q;
}
inline size_t gw_any_lds(const GwGeom& q, int T) {
    return std::max(static_cast<size_t>(q.bytes()), TXW * sizeof(float) * 256 * std::min((T + 255) / 256, GW_TILES));
}

// an element that three bf16 terms do not carry: its nearest bf16 is not finite
DEVINL bool beyond_terms(float x) { return (__float_as_uint(x) & 0x7fffffffu) >= 0x7f7f8000u; }
DEVINL bool beyond_terms(const float4& v) { return beyond_terms(v.x) | beyond_terms(v.y) | beyond_terms(v.z) | beyond_terms(v.w); }
// v = p[0] + p[1] + p[2], four elements as packed pairs
struct B3x4 { uint2 p[NPL]; };
DEVINL B3x4 split3x4(float4 v) {
    B3x4 r;
#pragma unroll
    for (int z = 0; z < NPL; ++z) {
        r.p[z] = make_uint2(pack_bf2(v.x, v.y), pack_bf2(v.z, v.w));
        v.x -= bf_lo(r.p[z].x); v.y -= bf_hi(r.p[z].x); v.z -= bf_lo(r.p[z].y); v.w -= bf_hi(r.p[z].y);
    }
    return r;
}
// whether any thread of the workgroup says so; red: one word, zeroed by thread 0 at least one barrier before; takes one barrier
DEVINL bool any_thread(bool x, int* red) {
    if (__ballot(x) != 0ull && (threadIdx.x & 63) == 0) *red = 1;
    __syncthreads();
    return *red != 0;
}

// threadIdx.x, hidden from the optimiser: it would keep the addresses of every piece across the loops of timex_gw_any, in scratch
DEVINL int own_thread() {
    int t = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(t));
    return t;
}
// Rows as 16-byte pieces, `per` a row: the thread's pieces tid + 512 i of `rows` rows are each(i, row, first step).
template <int NP, class F> DEVINL void for_pieces(int rows, int per, uint32_t per_inv, const F& each) {
    const int me = own_thread(), dr = over_per(TXT, per_inv), dt = 4 * (TXT - dr * per);
    int rr = over_per(me, per_inv), t = 4 * (me - rr * per);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        if (TXT * i >= rows * per) break;
        each(i, rr, t);
        rr += dr; t += dt;
        if (t >= 4 * per) { t -= 4 * per; ++rr; }
    }
}
// rows b0 .. b0 + q.bg - 1 of channel c
template <int NP> struct Stager {
    float4 x[NP];
    DEVINL void fetch(const float* __restrict__ in, const AnyGeom& q, int c, int b0, int B, int C, int T) {
#pragma unroll
        for (int i = 0; i < NP; ++i) x[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for_pieces<NP>(q.bg, 8 * q.nt, q.per_inv, [&](int i, int rr, int t) __attribute__((always_inline)) {
            if (rr < q.bg && b0 + rr < B && t < T) x[i] = *reinterpret_cast<const float4*>(in + (static_cast<size_t>(b0 + rr) * C + c) * T + t);
        });
    }
    DEVINL bool beyond() const {
        bool on = false;
#pragma unroll
        for (int i = 0; i < NP; ++i) on |= beyond_terms(x[i]);
        return on;
    }
    DEVINL void store(uint16_t* rp, const AnyGeom& q) const {
        const int pl = static_cast<int>(q.plane());
        for_pieces<NP>(q.bg, 8 * q.nt, q.per_inv, [&](int i, int rr, int t) __attribute__((always_inline)) {
            if (rr >= q.bg) return;
            uint16_t* d = rp + (q.zb + rr * q.pitch + (t >> 5)) * BLK + (t & 31);
            const B3x4 y = split3x4(x[i]);
#pragma unroll
            for (int p = 0; p < NPL; ++p) *reinterpret_cast<uint2*>(d + p * pl) = y.p[p];
        });
    }
};
// four elements at place `at` of a line (a multiple of 4) and one place further down in its second copy (nothing before its start)
DEVINL void put_line4(uint16_t* line, uint16_t* copy, int at, const uint2& y) {
    *reinterpret_cast<uint2*>(line + at) = y;
    if (at > 0) copy[at - 1] = static_cast<uint16_t>(y.x);
    *reinterpret_cast<uint32_t*>(copy + at) = (y.x >> 16) | (y.y << 16);
    copy[at + 2] = static_cast<uint16_t>(y.y >> 16);
}
// eight elements from the first (shift = 0) or second (16) of the dwords at x
DEVINL bf16x8 window8(const uint32_t* x, uint32_t shift) {
    uint32_t d[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) d[e] = x[e];
    return __builtin_bit_cast(bf16x8, make_uint4(__builtin_amdgcn_alignbit(d[1], d[0], shift), __builtin_amdgcn_alignbit(d[2], d[1], shift),
                                                 __builtin_amdgcn_alignbit(d[3], d[2], shift), __builtin_amdgcn_alignbit(d[4], d[3], shift)));
}
// the blocks in front of the first row and behind every row
DEVINL void zero_blocks(uint16_t* rp, const AnyGeom& q) {
    const int n = q.zb * (q.bg + 1) * (BLK / 8);
    const size_t pl = q.plane();
    for (int i = threadIdx.x; i < n; i += TXT) {
        const int blk = i / (BLK / 8), e = i - blk * (BLK / 8), row = over16(blk, q.zb_inv), z = blk - row * q.zb;      // row 0: the front
        uint16_t* d = rp + (row * q.pitch + z) * BLK + 8 * e;
#pragma unroll
        for (int p = 0; p < NPL; ++p) *reinterpret_cast<uint4*>(d + p * pl) = make_uint4(0, 0, 0, 0);
    }
}

// PAIRS: as the plan says; without, every tile has a wave of its own, the longest four on the four SIMDs
template <bool MIRROR, int COPIES, bool PAIRS>
__global__ __launch_bounds__(TXT, 4) void timex_conv_any(const float* __restrict__ w, const float* __restrict__ in, float* __restrict__ out,
                                                         float eps, int B, int C, int T, int ng, const ConvPlans plans) {
    extern __shared__ __align__(16) float lds[];
    // The first group of all channels, then the second ...: the larger groups come first, and every XCD gets some of each (by channels, with
    // two or four groups of two sizes, half of them got the larger ones only: B10 C768 T1500 130 us, 114 so; B5 C200 T388 9.1 / 7.7)
    const int grp = blockIdx.x / C, c = blockIdx.x - grp * C, fewer = B / ng, b0 = grp * fewer + min(grp, B % ng);
    const ConvPlan& plan = plans.p[grp < B % ng || B % ng == 0 ? 0 : 1];
    const AnyGeom& q = plan.q;
    const int Tp = 32 * q.nt, xl = h2_line_len(Tp), plane = static_cast<int>(q.plane());
    uint16_t* rp = reinterpret_cast<uint16_t*>(lds);                    // [NPL][plane]
    uint16_t* al = rp + NPL * plane;                                    // [NPL planes][COPIES][xl]
    int* red = reinterpret_cast<int*>(al + COPIES * NPL * xl);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, kh = lane >> 5;
    {
        Stager<CONV_PIECES> st;
        st.fetch(in, q, c, b0, B, C, T);
        float4 wr[T_ANY / (4 * TXT)];
#pragma unroll
        for (int z = 0; z < T_ANY / (4 * TXT); ++z) {
            const int tau = 4 * (z * TXT + tid);
            wr[z] = tau < T ? *reinterpret_cast<const float4*>(w + static_cast<size_t>(c) * T + tau) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        for (int i = tid; i < COPIES * NPL * xl / 8; i += TXT) reinterpret_cast<uint4*>(al)[i] = make_uint4(0, 0, 0, 0);
        zero_blocks(rp, q);
        if (tid == 0) *red = 0;
        bool beyond = st.beyond();
#pragma unroll
        for (int z = 0; z < T_ANY / (4 * TXT); ++z) beyond |= beyond_terms(wr[z]);
        __syncthreads();
        if (any_thread(beyond, red)) {
            for (int i = tid; i < q.bg * T; i += TXT) {
                const int b = i / T, t = i - b * T;
                const size_t row = (static_cast<size_t>(b0 + b) * C + c) * T;
                const float *x = in + row, *wl = w + static_cast<size_t>(c) * T + T - 1;       // wl[-lag]
                float acc = 0.f;
                if constexpr (MIRROR) { for (int s = t; s < T; ++s) acc = fmaf(wl[t - s], x[s], acc); }
                else { for (int s = 0; s <= t; ++s) acc = fmaf(wl[s - t], x[s], acc); }
                out[row + t] = MIRROR ? acc : acc + eps;
            }
            return;
        }
        st.store(rp, q);
        // tap tau (lag T-1-tau) sits at line position PZ + tau (forward) or 31 + lag (mirror); the rest is zero.  Four taps a thread: mirrored
        // they lie the other way round, an odd place up in the line and an even one in its second copy
#pragma unroll
        for (int z = 0; z < T_ANY / (4 * TXT); ++z) {
            const int tau = 4 * (z * TXT + tid);
            if (tau < T) {
                const B3x4 a = split3x4(MIRROR ? make_float4(wr[z].w, wr[z].z, wr[z].y, wr[z].x) : wr[z]);
#pragma unroll
                for (int p = 0; p < NPL; ++p) {
                    uint16_t *line = al + COPIES * p * xl, *copy = line + xl;
                    if constexpr (MIRROR) {
                        line += 28 + T - 4 - tau; copy += 28 + T - 4 - tau;          // (the lowest of the four at line[3], copy[2])
                        line[3] = static_cast<uint16_t>(a.p[p].x);
                        *reinterpret_cast<uint32_t*>(line + 4) = (a.p[p].x >> 16) | (a.p[p].y << 16);
                        line[6] = static_cast<uint16_t>(a.p[p].y >> 16);
                        if constexpr (COPIES == 2) {
                            *reinterpret_cast<uint32_t*>(copy + 2) = a.p[p].x;
                            *reinterpret_cast<uint32_t*>(copy + 4) = a.p[p].y;
                        }
                    } else if constexpr (COPIES == 2) put_line4(line, copy, PZ + tau, a.p[p]);
                    else *reinterpret_cast<uint2*>(line + PZ + tau) = a.p[p];
                }
            }
        }
        __syncthreads();
    }
    constexpr int TILES = PAIRS ? 2 : 1;
    const uint64_t pairs = PAIRS ? plan.pair : 0;
    const int pair = PAIRS ? ConvPlan::of(pairs, wv) : (wv < 4 ? wv : 11 - wv);
    const int ncol = q.nt * q.bg, ntile = (ncol + 31) >> 5;
    int tile[TILES], nd[TILES];
    const uint16_t* bp[TILES];
#pragma unroll
    for (int z = 0; z < TILES; ++z) {
        tile[z] = PAIRS && pair == NO_PAIR ? -1 : tile_of(ntile, MIRROR, TILES * pair + z);
        nd[z] = tile[z] < 0 ? 0 : tile_lags(q, MIRROR, tile[z]);
        const int col = min(32 * max(tile[z], 0) + ln, ncol - 1), a = over16(col, q.bg_inv), b = col - a * q.bg;
        bp[z] = rp + (q.zb + b * q.pitch + a) * BLK + 8 * kh;
    }
    const int d0 = PAIRS ? ConvPlan::of(plan.d0, wv) : 0, d1 = PAIRS ? ConvPlan::of(plan.d1, wv) : nd[0];
    const int start = (MIRROR ? 31 - ln : PZ + T - 1 - ln) + 8 * kh;    // forward: line[start - 32 d + j], mirror: line[start + 32 d + j]
    const uint32_t* ap = reinterpret_cast<const uint32_t*>(al + (COPIES == 2 ? start & 1 : 0) * xl) + (start >> 1);
    const uint32_t odd = 16 * (start & 1);
    f32x16 acc[TILES], low[TILES];  // the products of the first terms, which are what rounds; the other five
#pragma unroll
    for (int z = 0; z < TILES; ++z)
#pragma unroll
        for (int v = 0; v < 16; ++v) { acc[z][v] = 0.f; low[z][v] = 0.f; }
    auto run = [&](auto NTL, const int from, const int to) __attribute__((always_inline)) {
        constexpr int NT_ = decltype(NTL)::value;
        for (int d = from; d < to; ++d) {
            const int o = MIRROR ? d : -d;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                bf16x8 fa[NPL], fb[NT_][NPL];
#pragma unroll
                for (int p = 0; p < NPL; ++p) {
                    const uint32_t* a4 = ap + 16 * o + 8 * ks + p * (COPIES * xl >> 1);
                    if constexpr (COPIES == 2) fa[p] = __builtin_bit_cast(bf16x8, make_uint4(a4[0], a4[1], a4[2], a4[3]));
                    else fa[p] = window8(a4, odd);
                }
#pragma unroll
                for (int z = 0; z < NT_; ++z)
#pragma unroll
                    for (int p = 0; p < NPL; ++p)
                        fb[z][p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(bp[z] + BLK * o + 16 * ks + p * plane));
#pragma unroll
                for (int term = 0; term < 6; ++term)
#pragma unroll
                    for (int z = 0; z < NT_; ++z) {
                        f32x16& sum = term == 5 ? acc[z] : low[z];
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[TERM_A[term]], fb[z][TERM_B[term]], sum, 0, 0, 0);
                    }
            }
        }
    };
    if constexpr (PAIRS) {
        run(std::integral_constant<int, 2>{}, d0, min(d1, nd[1]));
        run(std::integral_constant<int, 1>{}, max(d0, nd[1]), d1);
        // the sums of a pair's other waves, through the LDS that the rows no longer need
        bool owner = pair != NO_PAIR;
        for (int x = 0; x < wv; ++x) owner &= ConvPlan::of(pairs, x) != pair;
        float4* const slot = reinterpret_cast<float4*>(lds);
        constexpr int SLOT4 = SUM_SLOT / 4;
        if (plan.shared) {
            __syncthreads();
            if (pair != NO_PAIR && !owner) {
#pragma unroll
                for (int z = 0; z < 2; ++z)
#pragma unroll
                    for (int v4 = 0; v4 < 4; ++v4)
                        slot[wv * SLOT4 + (4 * z + v4) * 64 + lane] = make_float4(acc[z][4 * v4] + low[z][4 * v4], acc[z][4 * v4 + 1] + low[z][4 * v4 + 1],
                                                                                 acc[z][4 * v4 + 2] + low[z][4 * v4 + 2], acc[z][4 * v4 + 3] + low[z][4 * v4 + 3]);
            }
            __syncthreads();
        }
        if (!owner) return;
        for (int x = wv + 1; x < TXW; ++x) {
            if (ConvPlan::of(pairs, x) != pair) continue;
#pragma unroll
            for (int z = 0; z < 2; ++z)
#pragma unroll
                for (int v4 = 0; v4 < 4; ++v4) {
                    const float4 y = slot[x * SLOT4 + (4 * z + v4) * 64 + lane];
                    acc[z][4 * v4] += y.x; acc[z][4 * v4 + 1] += y.y; acc[z][4 * v4 + 2] += y.z; acc[z][4 * v4 + 3] += y.w;
                }
        }
    } else {
        run(std::integral_constant<int, 1>{}, d0, d1);
    }
#pragma unroll
    for (int z = 0; z < TILES; ++z) {
        const int col = 32 * tile[z] + ln, a = over16(col, q.bg_inv), b = col - a * q.bg;
        if (tile[z] >= 0 && col < ncol) {
            float* o = out + (static_cast<size_t>(b0 + b) * C + c) * T;
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
                const int t = 32 * a + 8 * v4 + 4 * kh;
                float x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = (acc[z][4 * v4 + e] + low[z][4 * v4 + e]) + (MIRROR ? 0.f : eps);
                if (t < T) *reinterpret_cast<float4*>(o + t) = make_float4(x[0], x[1], x[2], x[3]);
            }
        }
    }
}

// the sum of a finished 32 x 32 tile of lag tile d over its diagonals, into diag[64 d ..] (entry l: lag 32 d + l - 31)
DEVINL void add_diagonals(float* diag, const f32x16& acc, int d, int ln, int kh) {
    float pos = 0.f, neg = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int t = 8 * (v >> 2) + 4 * kh + (v & 3);
        const float y = __shfl(acc[v], (kh << 5) | ((t - ln) & 31), 64);
        if (t >= ln) pos += y; else neg += y;
    }
    pos += __shfl_xor(pos, 32, 64);
    neg += __shfl_xor(neg, 32, 64);
    if (kh == 0) diag[64 * d + 31 + ln] += pos;
    else if (ln >= 1) diag[64 * d + ln - 1] += neg;
}

// The kernel gradient of short rows, where a tile of 256 lags is mostly empty (gw_plan): lag tiles of 32, M_d of columns (block, row) as in
// the convolution.  One workgroup: channel c = blockIdx.x, batch groups blockIdx.y, blockIdx.y + gridDim.y, ...; out[blockIdx.y][c][T]
__global__ __launch_bounds__(TXT, 4) void timex_gw_short(const float* __restrict__ k, const float* __restrict__ g, float* __restrict__ out,
                                                       int B, int C, int T, int ng, const AnyGeom q) {
    extern __shared__ __align__(16) float lds[];
    const int plane = static_cast<int>(q.plane());
    uint16_t* gp = reinterpret_cast<uint16_t*>(lds);            // [NPL][plane]
    uint16_t* kp = gp + NPL * plane;                            // [NPL][plane]
    float* diag = reinterpret_cast<float*>(kp + NPL * plane);   // [nt][64]
    int* red = reinterpret_cast<int*>(diag + 64 * q.nt);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, kh = lane >> 5, l16 = lane & 15;
    const int c = blockIdx.x, ncol = q.nt * q.bg, nsteps = (ncol + 15) >> 4;
    for (int i = tid; i < 64 * q.nt; i += TXT) diag[i] = 0.f;
    zero_blocks(gp, q);
    zero_blocks(kp, q);
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)gp));
    const uint32_t k_off = 2u * NPL * static_cast<uint32_t>(plane), pl_b = 2u * static_cast<uint32_t>(plane);
    const int db = 16 % q.bg, step_b = 2 * BLK * (db * q.pitch + 16 / q.bg), wrap_b = 2 * BLK * (1 - q.bg * q.pitch);
    for (int grp = blockIdx.y; grp < ng; grp += gridDim.y) {
        const int b0 = grp * q.bg;
        {
            Stager<GW_PIECES> sg, sk;
            sg.fetch(g, q, c, b0, B, C, T);
            sk.fetch(k, q, c, b0, B, C, T);
            __syncthreads();               // everybody is done with the group before
            if (tid == 0) *red = 0;
            __syncthreads();
            if (any_thread(sg.beyond() | sk.beyond(), red)) {
                for (int lag = tid; lag < T; lag += TXT) {
                    float acc = 0.f;
                    for (int b = b0; b < B && b < b0 + q.bg; ++b) {
                        const size_t row = (static_cast<size_t>(b) * C + c) * T;
                        for (int u = 0; u + lag < T; ++u) acc = fmaf(g[row + u + lag], k[row + u], acc);
                    }
                    diag[64 * (lag >> 5) + 31 + (lag & 31)] += acc;
                }
                continue;
            }
            sg.store(gp, q);
            sk.store(kp, q);
            __syncthreads();
        }
        // lag tile d takes the columns from d Bg on; tiles in the order of decreasing work go to the waves back and forth, two at
        // a time (their g operand is the same)
        for (int set = 0; 16 * set < q.nt; ++set) {
            const int dd[2] = {16 * set + wv, 16 * set + 15 - wv};
            if (dd[0] >= q.nt) break;
            f32x16 acc[2], low[2];          // as in timex_conv_any
#pragma unroll
            for (int z = 0; z < 2; ++z)
#pragma unroll
                for (int v = 0; v < 16; ++v) { acc[z][v] = 0.f; low[z][v] = 0.f; }
            int s = (dd[0] * q.bg) >> 4;
            // this lane's columns in the two transposing reads of a step: K slots 8 kh + (l16 >> 2) and four on
            int bb[2];
            uint32_t at[2];
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const int col = 16 * s + 8 * kh + (l16 >> 2) + 4 * z, a = over16(col, q.bg_inv);
                bb[z] = col - a * q.bg;
                at[z] = lds0 + 2u * static_cast<uint32_t>((q.zb + bb[z] * q.pitch + a) * BLK + 16 * (ln >> 4) + 4 * (l16 & 3));
            }
            auto operand = [&](const uint32_t o) __attribute__((always_inline)) {
                const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(at[0] + o));
                const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(at[1] + o));
                const uint2 x = __builtin_bit_cast(uint2, lo), y = __builtin_bit_cast(uint2, hi);
                return __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, y.x, y.y));
            };
            auto run = [&](auto NTL, const int end) __attribute__((always_inline)) {
                constexpr int NT_ = decltype(NTL)::value;
                for (; s < end; ++s) {
                    bf16x8 fg[NPL];
#pragma unroll
                    for (int p = 0; p < NPL; ++p) fg[p] = operand(p * pl_b);
                    bf16x8 fk[NT_][NPL];
#pragma unroll
                    for (int z = 0; z < NT_; ++z)
#pragma unroll
                        for (int p = 0; p < NPL; ++p) fk[z][p] = operand(k_off + p * pl_b - 2u * BLK * static_cast<uint32_t>(dd[z]));
#pragma unroll
                    for (int term = 0; term < 6; ++term)
#pragma unroll
                        for (int z = 0; z < NT_; ++z) {
                            f32x16& sum = term == 5 ? acc[z] : low[z];
                            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg[TERM_A[term]], fk[z][TERM_B[term]], sum, 0, 0, 0);
                        }
#pragma unroll
                    for (int z = 0; z < 2; ++z) {
                        at[z] += step_b; bb[z] += db;
                        if (bb[z] >= q.bg) { bb[z] -= q.bg; at[z] += wrap_b; }
                    }
                }
            };
            run(std::integral_constant<int, 1>{}, dd[1] < q.nt ? (dd[1] * q.bg) >> 4 : nsteps);
            run(std::integral_constant<int, 2>{}, nsteps);
#pragma unroll
            for (int z = 0; z < 2; ++z)
                if (dd[z] < q.nt) add_diagonals(diag, acc[z] + low[z], dd[z], ln, kh);     // a lag tile belongs to one wave
        }
    }
    __syncthreads();
    float* o = out + (static_cast<size_t>(blockIdx.y) * C + c) * T;
    for (int x = tid; x < T; x += TXT) {        // lag = 32 d + e comes from tile d (diagonal e) and tile d + 1 (diagonal e - 32)
        const int lag = T - 1 - x, d = lag >> 5, e = lag & 31;
        o[x] = diag[64 * d + 31 + e] + (d + 1 < q.nt ? diag[64 * (d + 1) + e - 1] : 0.f);
    }
}
// one workgroup: channel c = blockIdx.x, the batch rows of part blockIdx.y of gridDim.y, at most q.bg at a time; out[blockIdx.y][c][T]
__global__ __launch_bounds__(TXT, 4) void timex_gw_any(const float* __restrict__ k, const float* __restrict__ g, float* __restrict__ out,
                                                       int B, int C, int T, const GwGeom q) {
    extern __shared__ __align__(16) float lds[];
    uint16_t* gp = reinterpret_cast<uint16_t*>(lds);            // [bg][NPL][plane]
    int* red = reinterpret_cast<int*>(gp + q.bg * NPL * q.plane);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, kg = lane >> 4;
    const int c = blockIdx.x, np = gridDim.y, fewer = B / np, more = B % np, part = blockIdx.y;
    const int first = part * fewer + min(part, more), last = first + fewer + (part < more ? 1 : 0);
    const int bg = (last - first + (last - first + q.bg - 1) / q.bg - 1) / ((last - first + q.bg - 1) / q.bg);      // rows at a time, dealt evenly
    float* const o = out + (static_cast<size_t>(part) * C + c) * T;
    // nothing writes to the zeros around the rows again
    for (int i = tid; i < bg * NPL * q.plane / 8; i += TXT) reinterpret_cast<uint4*>(lds)[i] = make_uint4(0, 0, 0, 0);
    constexpr int NP = GW_PIECES;
    const int per = 8 * q.nt;
    float4 xg[NP], xk[NP];
    auto fetch = [&](const int b0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NP; ++i) xg[i] = xk[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for_pieces<NP>(bg, per, q.per_inv, [&](int i, int rr, int t) __attribute__((always_inline)) {
            if (rr < bg && b0 + rr < last && t < T) {
                const size_t at = (static_cast<size_t>(b0 + rr) * C + c) * T + t;
                xg[i] = *reinterpret_cast<const float4*>(g + at);
                xk[i] = *reinterpret_cast<const float4*>(k + at);
            }
        });
    };
    fetch(first);
    if (tid == 0) *red = 0;
    // what this wave adds up: lag tiles q0 .. q0 + nq - 1, every nw-th of the steps that they have
    const int all = (T + 255) >> 8;
    const bool wide = all > GW_TILES, second = wide && wv >= GW_WAVES;
    const int q0 = second ? GW_TILES : 0, nq = min(all - q0, GW_TILES), nw = wide ? (second ? TXW - GW_WAVES : GW_WAVES) : TXW;
    const int steps = q.nt - 8 * q0;
    f32x4 acc[GW_TILES], low[GW_TILES];          // as in timex_conv_any
#pragma unroll
    for (int z = 0; z < GW_TILES; ++z)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[z][v] = low[z][v] = 0.f;
    // g[t + (i & 7) + 128 (i >> 3)], K slots t = 8 kg ..; k[t - 8 j]
    const uint32_t* const ga = reinterpret_cast<const uint32_t*>(gp) + (((l16 & 7) + GW_OVER * (l16 >> 3) + 8 * kg) >> 1) + GW_OVER * q0;
    const uint32_t odd = 16 * (l16 & 1);
    const uint16_t* const ka = gp + q.k + 8 * kg - 8 * l16;
    bool fell = false;
    for (int b0 = first; b0 < last; b0 += bg) {
        bool beyond = false;
#pragma unroll
        for (int i = 0; i < NP; ++i) beyond |= beyond_terms(xg[i]) | beyond_terms(xk[i]);
        __syncthreads();               // everybody is done with the group before
        const bool loop = any_thread(beyond, red);
        if (loop) {
            for (int lag = tid; lag < T; lag += TXT) {
                float a = fell ? o[T - 1 - lag] : 0.f;
                for (int b = b0; b < last && b < b0 + bg; ++b) {
                    const size_t row = (static_cast<size_t>(b) * C + c) * T;
                    for (int u = 0; u + lag < T; ++u) a = fmaf(g[row + u + lag], k[row + u], a);
                }
                o[T - 1 - lag] = a;    // (read again by this thread alone)
            }
            fell = true;
        } else {
            for_pieces<NP>(bg, per, q.per_inv, [&](int i, int rr, int t) __attribute__((always_inline)) {
                if (rr >= bg) return;
                const B3x4 yg = split3x4(xg[i]), yk = split3x4(xk[i]);
                uint16_t* d = gp + rr * NPL * q.plane + GW_OVER * (t >> 7);
                uint16_t* dk = gp + rr * NPL * q.plane + q.k + t;
                const int r = t & 127;
                const bool twice = r < GW_OVER - 128 && t >= 128;
                static_assert(GW_OVER == 128 + 16, "");
#pragma unroll
                for (int p = 0; p < NPL; ++p, d += q.plane, dk += q.plane) {
                    *reinterpret_cast<uint2*>(d + r) = yg.p[p];
                    if (twice) *reinterpret_cast<uint2*>(d + r - 16) = yg.p[p];        // at the end of the block before
                    *reinterpret_cast<uint2*>(dk) = yk.p[p];
                }
            });
        }
        if (b0 + bg < last) fetch(b0 + bg);
        __syncthreads();
        if (tid == 0) *red = 0;
        if (loop || steps <= 0) continue;
        const int rows = min(bg, last - b0);
        int s = second ? wv - GW_WAVES : wv, row = 0;
        for (; s >= steps; s -= steps) ++row;
        while (row < rows) {
            const uint32_t* a4 = ga + (row * NPL * q.plane >> 1) + (GW_OVER / 2) * (s >> 2) + 16 * (s & 3);
            const uint16_t* b8 = ka + row * NPL * q.plane + 32 * s;
            const int on = min(nq, (s >> 3) + 1);
            bf16x8 fa[NPL];
#pragma unroll
            for (int p = 0; p < NPL; ++p, a4 += q.plane >> 1) {
                fa[p] = window8(a4, odd);
            }
#pragma unroll
            for (int z = 0; z < GW_TILES; ++z)
                if (z < on) {
                    bf16x8 fb[NPL];
#pragma unroll
                    for (int p = 0; p < NPL; ++p) fb[p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(b8 + p * q.plane - 256 * z));
#pragma unroll
                    for (int term = 0; term < 6; ++term) {
                        f32x4& sum = term == 5 ? acc[z] : low[z];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[TERM_A[term]], fb[TERM_B[term]], sum, 0, 0, 0);
                    }
                }
            for (s += nw; s >= steps; s -= steps) ++row;
        }
    }
    // the waves' sums, in their order, through the LDS that the rows no longer need
    __syncthreads();
    f32x4* const slot = reinterpret_cast<f32x4*>(lds);
    const int slots = min(all, GW_TILES);
#pragma unroll
    for (int z = 0; z < GW_TILES; ++z)
        if (z < nq) slot[(wv * slots + z) * 64 + lane] = acc[z] + low[z];
    __syncthreads();
    for (int lag = tid; lag < T; lag += TXT) {
        const int r = lag & 255, i = (r & 7) + 8 * (r >> 7), z = lag >> 8;
        const bool up = z >= GW_TILES;
        const int w0 = up ? GW_WAVES : 0, w1 = wide && !up ? GW_WAVES : TXW;
        const float* x = lds + (w0 * slots + (up ? z - GW_TILES : z)) * 256 + (16 * (i >> 2) + ((r >> 3) & 15)) * 4 + (i & 3);
        float sum = fell ? o[T - 1 - lag] : 0.f;
        for (int w = w0; w < w1; ++w, x += 256 * slots) sum += *x;
        o[T - 1 - lag] = sum;
    }
}
// out[x] = sum of n parts that lie `size` floats apart, four elements a thread
__global__ __launch_bounds__(256) void timex_add_parts(const float4* __restrict__ part, float4* __restrict__ out, size_t size4, int n) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= size4) return;
    float4 a = part[i];
    for (int z = 1; z < n; ++z) {
        const float4 x = part[i + z * size4];
        a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
    }
    out[i] = a;
}

// The waves' shares: runs of a pair's lags are added where the longest run is, until there are eight or a run would have less than RUN_MIN
// steps (of a tile and a lag; so many take about what it takes to add two waves' sums), then the longest four runs go to the
// four SIMDs (a wave w runs on SIMD w mod 4) and the others to the least loaded ones.  The plans of a call take 0.15 to 1.0 us of host time.
constexpr int RUN_MIN = 4;
// returns how many more steps the longest tile has than the longest run, 0 at least; large: more tiles than waves
int plan_waves(ConvPlan& p, bool mirror) {
    const int ntile = (p.q.nt * p.q.bg + 31) / 32, npair = (ntile + 1) / 2;
    int lags[TXW][2] = {}, runs[TXW] = {}, work[TXW] = {};
    for (int m = 0; m < npair; ++m) {
        for (int z = 0; z < 2; ++z) {
            const int t = tile_of(ntile, mirror, 2 * m + z);
            lags[m][z] = t < 0 ? 0 : tile_lags(p.q, mirror, t);
        }
        work[m] = lags[m][0] + lags[m][1];
        runs[m] = 1;
    }
    for (int n = npair; n < TXW; ++n) {
        int most = -1;
        for (int m = 0; m < npair; ++m)
            if (work[m] >= RUN_MIN * (runs[m] + 1) && (most < 0 || work[m] * runs[most] > work[most] * runs[m])) most = m;
        if (most < 0) break;
        ++runs[most];
    }
    struct Run { int pair, d0, d1, work; } run[TXW];
    int n = 0;
    for (int m = 0; m < npair; ++m) {
        const auto lag_at = [&](int x) { return x < 2 * lags[m][1] ? (x + 1) / 2 : x - lags[m][1]; };      // after x steps of the pair
        for (int k = 0; k < runs[m]; ++k) {
            const int d0 = lag_at(work[m] * k / runs[m]), d1 = k + 1 == runs[m] ? lags[m][0] : lag_at(work[m] * (k + 1) / runs[m]);
            if (d1 > d0) run[n++] = {m, d0, d1, (d1 - d0) + (d0 < lags[m][1] ? (d1 < lags[m][1] ? d1 : lags[m][1]) - d0 : 0)};
        }
    }
    std::sort(run, run + n, [](const Run& a, const Run& b) { return a.work > b.work; });
    p.shared = n > npair;
    p.pair = ~uint64_t{0};
    p.d0 = p.d1 = 0;
    for (int i = 0; i < n; ++i) {
        const int at = 8 * (i < 4 ? i : 11 - i);
        p.pair ^= static_cast<uint64_t>(NO_PAIR ^ run[i].pair) << at;
        p.d0 |= static_cast<uint64_t>(run[i].d0) << at;
        p.d1 |= static_cast<uint64_t>(run[i].d1) << at;
    }
    return ntile > TXW ? 1 << 20 : std::max(0, tile_lags(p.q, mirror, tile_of(ntile, mirror, 0)) - run[0].work);
}
size_t conv_plan_lds(const ConvPlans& x) {
    return std::max({conv_any_lds(x.p[0].q, x.copies), conv_any_lds(x.p[1].q, x.copies), x.p[0].shared || x.p[1].shared ? TXW * SUM_SLOT * sizeof(float) : 0});
}
// A wave a tile is what short rows take, up to SHORT_ROWS steps, where the longest tile has no more than so many steps over the longest run: an
// instance without sums through LDS, without the plan's bytes and with the accumulators of one tile, in half the registers, so that three or four
// workgroups share a CU; fewer steps where the rows' LDS has room for two only, and where a CU has one workgroup at most, which waits for its
// longest wave.  A convolution, us, as runs / a wave a tile: B16 C768 T132 11.3 / 8.3, B32 C1000 T60 10.8 / 7.9, B3 C768 T452 14.1 / 11.5, B4 C1000 T484
// (12 steps) 17.0 / 13.2, B3 C640 T644 (17) 14.9 / 12.5; two by LDS: B10 C640 T580 (8) 21.7 / 22.7; few workgroups: B1 C64 T260 (4) 5.5 / 6.4.
constexpr int TILE_STEPS = 16, TILE_STEPS_FULL = 5, TILE_STEPS_FEW = 3;
constexpr int SHORT_ROWS = 672;        // (B13 C300 T772 25.2 / 26.6)
// Batch rows of a unit, dealt evenly to `ng` units a channel.  What finishes first by a count of matrix clocks (96 per column tile and
// block lag on a CU's four SIMDs), conversion and a fixed cost, in rounds of two workgroups per CU; at most 16 tiles (a pair a wave) and
// 80 KB.  Units of two sizes count by their mean, but in the last round by the larger: B3 C200 T644 as 2 + 1 rows, one round, 9.2 us, as
// 1 + 1 + 1, two rounds of half the time, 8.1; B9 C200 T196 7.0 / 5.9.  A last round after others that leaves every CU one workgroup at most, which
// then runs nearly twice as fast, counts three quarters: B3 C768 T1500 as 3 rows, 1.5 rounds, 36.0 us, as 2 + 1, three, 44.6; B19 C640 T772 50.7 / 56.6.
ConvPlans conv_any_plans(int B, int C, int T, bool mirror, int* ng) {
    ConvPlans best{};
    double cost = 1e300;
    for (int most = 1; most <= B && most <= 32; ++most) {
        const int groups = (B + most - 1) / most, rows[2] = {(B + groups - 1) / groups, B / groups};
        if (rows[0] != most) continue;
        ConvPlans x{};
        double unit = 0, largest = 0;
        for (int z = 0; z < 2; ++z) {
            x.p[z].q = any_geom(T, rows[z], 31);
            const int ntile = (x.p[z].q.nt * rows[z] + 31) / 32;
            if (ntile > 2 * TXW) { unit = -1; break; }
            const int share = z == 1 ? groups - B % groups : B % groups;
            long long steps = 0;
            for (int t = 0; t < ntile; ++t) steps += tile_lags(x.p[z].q, mirror, t);
            const double one = 96.0 * steps + 0.15 * rows[z] * T + 3000.0;
            if (z == 0) largest = one;
            unit += one * share / groups;
        }
        x.copies = most == 1 && conv_any_lds(x.p[0].q, 2) > LDS_ANY ? 1 : 2;
        if (unit < 0 || conv_plan_lds(x) > LDS_ANY || 8 * x.p[0].q.nt * rows[0] > CONV_PIECES * TXT) { if (most > 1) break; }
        const long long units = static_cast<long long>(C) * groups, full = (units - 1) / (2 * NCU);
        const double c = full * unit + (full > 0 && units - full * 2 * NCU <= NCU ? 0.75 : 1.0) * largest;
        if (c < cost) { cost = c; best = x; *ng = groups; }
    }
    int longer = 0;
    for (ConvPlan& p : best.p) longer = std::max(longer, plan_waves(p, mirror));
    const bool room = 3 * std::max(conv_any_lds(best.p[0].q, best.copies), conv_any_lds(best.p[1].q, best.copies)) <= LDS_CU;
    best.pairs = T > SHORT_ROWS || longer > (static_cast<long long>(C) * *ng <= 2 * NCU ? TILE_STEPS_FEW : (room ? TILE_STEPS : TILE_STEPS_FULL));
    if (!best.pairs) best.p[0].shared = best.p[1].shared = 0;
    return best;
}
inline size_t gw_short_lds(const AnyGeom& q) { return 2 * NPL * q.plane() * 2 + static_cast<size_t>(q.nt) * 256 + 16; }
AnyGeom gw_short_geom(int B, int T) {
    AnyGeom best = any_geom(T, 1, 15);
    for (int bg = 2; bg <= B && bg <= 32; ++bg) {
        const AnyGeom q = any_geom(T, bg, 15);
        if (gw_short_lds(q) > LDS_ANY || 8 * q.nt * bg > GW_PIECES * TXT) break;
        best = q;
    }
    return best;
}
// as many rows at a time as leave room for two workgroups per CU
GwGeom gw_any_geom(int B, int T) {
    GwGeom best = gw_geom(T, 1);
    for (int bg = 2; bg <= B && bg <= 32; ++bg) {
        const GwGeom q = gw_geom(T, bg);
        if (gw_any_lds(q, T) > LDS_ANY || 8 * q.nt * bg > GW_PIECES * TXT) break;
        best = q;
    }
    return best;
}
// What the kernel gradient does: lag tiles of 32 (timex_gw_short) or of 256, and how many parts of the batch side by side (their sums are added
// by a second kernel).
struct GwPlan { bool narrow; int parts; };
// Batch groups of timex_gw_short side by side: as many as it takes for two workgroups per CU.
int gw_group_parts(int B, int C, int T) {
    const int bg = gw_short_geom(B, T).bg, ng = (B + bg - 1) / bg, want = (2 * NCU + C - 1) / C;
    return ng < want ? ng : want;
}
int gw_most_parts(int B, int C) { return std::max(1, std::min(B, 8 * NCU / C)); }
// Parts for timex_gw_any by a count of clocks, in rounds of two workgroups per CU: 48 a row, step and lag tile, 3 a row and step of time for its
// conversion, a fixed cost a workgroup and that of the second kernel.
int gw_clock_parts(int B, int C, int T) {
    const int nt = (T + 31) / 32;
    long long row = 3LL * T;
    for (int s = 0; s < nt; s += 8) row += 48LL * (nt - s);
    int best = 1;
    long long cost = -1;
    for (int p = 1; p <= gw_most_parts(B, C); ++p) {
        const long long x = (static_cast<long long>(C) * p + 2 * NCU - 1) / (2 * NCU) * (12000 + row * B / p) + (p > 1 ? 10000 : 0);
        if (cost < 0 || x < cost) { cost = x; best = p; }
    }
    return best;
}
// Up to GW_SHORT steps lag tiles of 32, a tile of 256 being mostly empty: the kernel alone, 32 / 256, B32 C1000 T36 12.7 / 16.2 us, B20 C700 T260 27.6 /
// 27.7.  Up to GW_MIDDLE what takes less by the formulas below, us fitted to 5400 timings of both with one to sixteen parts (B2 to B32, C64 to
// C1000, T388 to T708; they are off by 4 % rms): timex_gw_short's whole groups of rows, of which one or two fit a small batch, and its fewer
// workgroups against timex_gw_any's parts.  Backward, 32 / 256 with the formula's parts / with those by clocks: B24 C300 T484 46.3 / 48.0 / 52.2 us, B8
// C200 T484 17.7 / 19.2 / 20.2, B20 C1000 T388 74.0 / 79.6 / 80.1, B12 C768 T452 53.5 / 48.3 / 48.1.  Up to GW_FITTED, where the timings end, the parts
// are the formula's, too (B6 C200 T644 23.0 -> 21.7); beyond, by clocks (B7 C300 T1500 74 us, 81 by the formula).
constexpr int GW_SHORT = 384, GW_MIDDLE = 512, GW_FITTED = 708;
GwPlan gw_plan(int B, int C, int T) {
    const int groups = gw_group_parts(B, C, T);
    if (T <= GW_SHORT) return {true, groups};
    if (T > GW_FITTED) return {false, gw_clock_parts(B, C, T)};
    const auto over = [](long long x, long long d) { return static_cast<double>((x + d - 1) / d); };
    const int nt = (T + 31) / 32, bg = gw_any_geom(B, T).bg;
    double steps = 0, cost = 1e300;
    for (int s = 0; s < nt; s += 8) steps += nt - s;
    GwPlan best{false, 1};
    for (int p = 1; p <= gw_most_parts(B, C); ++p) {
        const long long w = static_cast<long long>(C) * p, rows = (B + p - 1) / p;
        const double x = 1.41 * over(w, 2 * NCU) * over(rows, bg) + rows * steps * (0.0141 * over(w, NCU) + 0.011 * over(w, 2 * NCU)) + (p > 1 ? 1.13 + 5.2e-6 * w * T : 0.0);
        if (x < cost) { cost = x; best.parts = p; }
    }
    if (T <= GW_MIDDLE) {
        const int rows = gw_short_geom(B, T).bg;
        const long long w = static_cast<long long>(C) * groups;
        const double per = over(over(B, rows), groups);
        if (over(w, 2 * NCU) * (0.55 + 1.61 * per) + 0.00144 * over(w, NCU) * per * rows * nt * nt + (groups > 1 ? 0.95 : 0.0) < cost) return {true, groups};
    }
    return best;
}

constexpr int T_MAX = 4096;

int check_tx(int B, int C, int T) {
    if (B <= 0 || C <= 0 || T <= 0) return RWKV_ERR_SHAPE;
    if (T % 4 != 0 || T > T_MAX) return RWKV_ERR_SHAPE;
    if (B > 8 * 65535) return RWKV_ERR_SHAPE;
    return RWKV_OK;
}

// Whole tiles of steps and enough batch rows for the 32 columns of a product: the kernels whose operands are shared best.  B32
// C768 T768 forward: 58 us here, 64 with the kernel for any shape.
bool use_mfma(int B, int T) { return T % 32 == 0 && T <= T_MFMA_MAX && B >= 8; }
int conv_grid(int B, int C) {
    const long long units = static_cast<long long>(C) * ((B + MROWS - 1) / MROWS);
    return static_cast<int>(units < NCU ? units : NCU);
}

template <typename K> int raise_lds_limit(K kernel, size_t bytes) {
    if (bytes <= 48 * 1024) return RWKV_OK;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess) { g_last_hip_error = static_cast<int>(e); return RWKV_ERR_LAUNCH; }
    return RWKV_OK;
}

}  // namespace
}  // namespace rwkv

using namespace rwkv;

// the convolution (forward) or its mirror (gk = the mirrored convolution of gwk with w)
template <bool MIRROR> int launch_conv(void* stream, const float* w, const float* in, float* out, float eps, int B, int C, int T) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (use_mfma(B, T)) {
        const size_t lds = h2_lds_bytes(T);
        auto kernel = T <= T_H2_MID ? timex_conv_h2<MIRROR, T_H2_MID / 256> : timex_conv_h2<MIRROR, T_H2_MAX / 256>;
        if (int e = raise_lds_limit(kernel, lds)) return e;
        hipLaunchKernelGGL(kernel, dim3(conv_grid(B, C)), dim3(TXT), lds, st, w, in, out, eps, B, C, T);
    } else {
        int ng;
        const ConvPlans plans = conv_any_plans(B, C, T, MIRROR, &ng);
        const size_t lds = conv_plan_lds(plans);
        if (static_cast<long long>(C) * ng > 0x7fffffffLL) return RWKV_ERR_SHAPE;
        const auto kernel = !plans.pairs ? timex_conv_any<MIRROR, 2, false> : (plans.copies == 2 ? timex_conv_any<MIRROR, 2, true> : timex_conv_any<MIRROR, 1, true>);
        if (int e = raise_lds_limit(kernel, lds)) return e;
        hipLaunchKernelGGL(kernel, dim3(C * ng), dim3(TXT), lds, st, w, in, out, eps, B, C, T, ng, plans);
    }
    return RWKV_OK;
}

extern "C" {

int rwkv_timex_forward(void* stream, const float* w, const float* k, float* x, float eps, int B, int C, int T) {
    if (int e = check_tx(B, C, T)) return e;
    if (int e = check_ptrs({w, k, x})) return e;
    if (int e = launch_conv<false>(stream, w, k, x, eps, B, C, T)) return e;
    return launch_status();
}

int rwkv_timex_backward(void* stream, const float* w, const float* k, const float* gwk, float* gw, float* gk,
                        int B, int C, int T) {
    if (int e = check_tx(B, C, T)) return e;
    if (int e = check_ptrs({w, k, gwk, gw, gk})) return e;
    if (static_cast<long long>(B) * C > 0x7fffffffLL) return RWKV_ERR_SHAPE;
    if (int e = launch_conv<true>(stream, w, gwk, gk, 0.0f, B, C, T)) return e;
    hipLaunchKernelGGL(timex_gw, dim3(B * C), dim3(T / 4), (2 * static_cast<size_t>(T) + 4) * sizeof(float),
                       static_cast<hipStream_t>(stream), k, gwk, gw, T);
    return launch_status();
}

int rwkv_timex_backward_sum(void* stream, const float* w, const float* k, const float* gwk, float* gw_sum, float* gk,
                            int B, int C, int T) {
    if (int e = check_tx(B, C, T)) return e;
    if (T % 32 != 0 || T > T_MFMA_MAX) return RWKV_ERR_SHAPE;
    if (int e = check_ptrs({w, k, gwk, gw_sum, gk})) return e;
    if (int e = launch_conv<true>(stream, w, gwk, gk, 0.0f, B, C, T)) return e;
    // (any batch size: a pass takes 16 rows, rows past the batch count as zero)
    const size_t lds_gw = gw_h2_lds_bytes(T);
    auto kernel = T <= T_H2_MID ? timex_gw_sum_h2<T_H2_MID / 256> : timex_gw_sum_h2<T_H2_MAX / 256>;
    if (int e = raise_lds_limit(kernel, lds_gw)) return e;
    hipLaunchKernelGGL(kernel, dim3(C < NCU ? C : NCU), dim3(TXT), lds_gw, static_cast<hipStream_t>(stream), k, gwk, gw_sum, B, C, T);
    return launch_status();
}

size_t rwkv_timex_backward_ws_bytes(int B, int C, int T) {
    if (check_tx(B, C, T) != RWKV_OK || (T % 32 == 0 && T <= T_MFMA_MAX)) return 0;
    const int parts = gw_plan(B, C, T).parts;
    return parts <= 1 ? 0 : static_cast<size_t>(parts) * C * T * sizeof(float);
}

int rwkv_timex_backward_ws(void* stream, const float* w, const float* k, const float* gwk, float* gw_sum, float* gk, int B, int C, int T,
                           void* workspace, size_t workspace_bytes) {
    if (int e = check_tx(B, C, T)) return e;
    if (T % 32 == 0 && T <= T_MFMA_MAX) return rwkv_timex_backward_sum(stream, w, k, gwk, gw_sum, gk, B, C, T);
    if (int e = check_ptrs({w, k, gwk, gw_sum, gk})) return e;
    // a workspace with room for fewer parts is for timex_gw_any, which takes any number of them (without room: one, in gw_sum itself); too few to
    // fill the card, as all rules for their number have it, are refused
    GwPlan plan = gw_plan(B, C, T);
    const int groups = gw_group_parts(B, C, T), least = T <= GW_SHORT ? groups : std::min({plan.parts, groups, gw_clock_parts(B, C, T)});
    const size_t room = workspace != nullptr && aligned16(workspace) ? workspace_bytes / (static_cast<size_t>(C) * T * sizeof(float)) : 0;
    if (least > 1 && room < static_cast<size_t>(least)) return RWKV_ERR_WORKSPACE;
    if (plan.parts > 1 && room < static_cast<size_t>(plan.parts)) plan = {false, room > 1 ? static_cast<int>(room) : 1};
    const int parts = plan.parts;
    if (int e = launch_conv<true>(stream, w, gwk, gk, 0.0f, B, C, T)) return e;
    hipStream_t st = static_cast<hipStream_t>(stream);
    float* const to = parts > 1 ? static_cast<float*>(workspace) : gw_sum;
    if (plan.narrow) {
        const AnyGeom q = gw_short_geom(B, T);
        const size_t lds = gw_short_lds(q);
        if (int e = raise_lds_limit(timex_gw_short, lds)) return e;
        hipLaunchKernelGGL(timex_gw_short, dim3(C, parts), dim3(TXT), lds, st, k, gwk, to, B, C, T, (B + q.bg - 1) / q.bg, q);
    } else {
        const GwGeom q = gw_any_geom(B, T);
        const size_t lds = gw_any_lds(q, T);
        if (int e = raise_lds_limit(timex_gw_any, lds)) return e;
        hipLaunchKernelGGL(timex_gw_any, dim3(C, parts), dim3(TXT), lds, st, k, gwk, to, B, C, T, q);
    }
    if (parts > 1) {
        const size_t n4 = static_cast<size_t>(C) * T / 4;
        hipLaunchKernelGGL(timex_add_parts, dim3(static_cast<unsigned>((n4 + 255) / 256)), dim3(256), 0, st,
                           static_cast<const float4*>(workspace), reinterpret_cast<float4*>(gw_sum), n4, parts);
    }
    return launch_status();
}

}  // extern "C"
