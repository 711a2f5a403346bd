// wkv6 / wkv6_state (raw bf16 decay) and wkv5 (one decay per channel), head size 64, sequences cut into blocks of time: what a block
// makes of a state that enters it empty, and the log2 of its decay per key channel.  Up to SCAN_BLOCKS blocks are chained by the kernels that start
// from them (wkv6_fwd_f.hip, wkv6_bwd_f.hip), more by wkv6_scan (wkv6_fwd_f.hip).
//     forward   E[i][j] = sum_t v_t[i] k_t[j] 2^{sum of the decays after t}          backward  sum_t gy_t[i] r_t[j] 2^{sum of the decays before t}
// Nothing but this sum comes out of a block, so it is no chain of chunks: the tokens' exponents are direct sums of log decays (never above
// zero: nothing overflows, and whatever a decay is it needs no second path), and E is one product over up to SUP tokens at a time.
//
// One workgroup of sixteen waves per (batch, head, block).  A wave takes 16 tokens, a lane two neighbouring channels of eight of them (128-byte
// rows): its decays' sums go to LDS, then each wave adds up what lies between its tokens and the end, and leaves K'' as hi and lo bf16
// planes beside the values'.  Then a wave makes one 16 x 16 tile of E.  B1 H32 T3001, 8 blocks of 384 tokens: forward 17.5 -> 13.1 us, backward
// 18.4 -> 13.1, against the kernels that go on from there run without outputs, which walk through the chunks and fill a pipeline first;
// it clears the flag words too, a launch of its own before.  The launch takes 4 of the 13, its 37 MB 7 at a copy's rate.
#include "wkv6_fused.h"

namespace rwkv {
namespace {

constexpr int SUP = 256, NTL = 1024;
constexpr lds_t ROWL = 144, PLANEL = SUP * ROWL;

struct ArgsL {
    int T, C, H, NB, TB;
    const uint16_t *key, *val, *w;
    float *state, *decay;              // [B*H][NB][64][64], [B*H][NB][64]
    int* flags;                        // [B*H][8], cleared: the kernels that follow only set them
};
struct SmemL {
    uint16_t plane[3][SUP][ROWL / 2];  // K'' hi, lo, V
    float sums[16][N], total[N];
};

template <bool REV, bool HD>
__global__ __launch_bounds__(NTL) void wkv6_local(const ArgsL a) {
    __shared__ SmemL S;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bh = __builtin_amdgcn_readfirstlane(blockIdx.x / a.NB), blk = blockIdx.x - bh * a.NB;
    const int b = __builtin_amdgcn_readfirstlane(bh / a.H), h = bh - b * a.H;
    if (blk == 0 && tid < 8) a.flags[bh * 8 + tid] = 0;
    if (REV ? blk == 0 : blk == a.NB - 1) return;                        // (nobody asks what leaves the last block)
    if constexpr (HD)
        if (strong_layer(a.w, a.C, lane)) return;                        // wkv5_bf.hip does the layer
    const int t0 = blk * a.TB, len = min(a.TB, a.T - t0);
    const int parts = (len + SUP - 1) / SUP, per = ((len + parts - 1) / parts + 31) / 32 * 32;      // tokens at a time
    const size_t base = (static_cast<size_t>(b) * a.T + t0) * a.C + static_cast<size_t>(h) * N;
    const int half = lane >> 5, p = lane & 31, tk = 16 * wv + 8 * half;  // the lane's tokens tk .. tk + 7, channels 2 p, 2 p + 1
    const int vrow = 16 * wv + (lane >> 3), vpc = lane & 7;              // rows vrow, vrow + 8 of the values, 16 bytes vpc
    const lds_t sb = lds_of(&S);
    float lamc[2] = {0.f, 0.f};
    if constexpr (HD) {
        const uint32_t x = *reinterpret_cast<const uint32_t*>(a.w + h * N + 2 * p);
        lamc[0] = -LOG2E * exp2_fast(LOG2E * bf_lo(x)); lamc[1] = -LOG2E * exp2_fast(LOG2E * bf_hi(x));
    }
    uint32_t xk[8], xw[8];
    uint4 xv[2];
    const bool on = 16 * wv < per;
    // (a uniform base and a 32-bit byte offset a lane, clamped to the block's last token; below 2^31 bytes a batch row)
    const uint32_t row_b = 2u * static_cast<uint32_t>(a.C), end = static_cast<uint32_t>(len - 1) * row_b;
    const char* const pk = reinterpret_cast<const char*>(a.key + base);
    const char* const pw = reinterpret_cast<const char*>(a.w + (HD ? 0 : base));
    const char* const pv = reinterpret_cast<const char*>(a.val + base);
    const uint32_t ok = static_cast<uint32_t>(tk) * row_b, ov = static_cast<uint32_t>(vrow) * row_b;
    auto fetch = [&](const int part) __attribute__((always_inline)) {
        if (!on) return;
        const uint32_t s = static_cast<uint32_t>(part * per) * row_b;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t o = min(ok + (s + e * row_b), end) + 4 * p;
            xk[e] = *reinterpret_cast<const uint32_t*>(pk + o);
            if constexpr (!HD) xw[e] = *reinterpret_cast<const uint32_t*>(pw + o);
        }
#pragma unroll
        for (int z = 0; z < 2; ++z) xv[z] = *reinterpret_cast<const uint4*>(pv + (min(ov + (s + 8 * z * row_b), end) + 16 * vpc));
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float logd[2] = {0.f, 0.f};
    const int l16 = lane & 15, g = lane >> 4, it = wv >> 2, jt = wv & 3;
    fetch(REV ? parts - 1 : 0);
    if (!on) {                                           // rows that no part has
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int q = 0; q < 3; ++q) lds_st<u32x4>(sb + q * PLANEL + (vrow + 8 * z) * ROWL + 16 * vpc, u32x4{0u, 0u, 0u, 0u});
    }
#pragma unroll 1
    for (int i = 0; i < parts; ++i) {
        const int part = REV ? parts - 1 - i : i, live = min(per, len - part * per);      // tokens of this part
        float lam[8][2], tot[2] = {0.f, 0.f}, other[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            // (masks, also below: of conditions the compiler makes branches)
            const uint32_t in = static_cast<uint32_t>((tk + e - live) >> 31);
            const float x0 = HD ? lamc[0] : -LOG2E * exp2_fast(LOG2E * bf_lo(xw[e])), x1 = HD ? lamc[1] : -LOG2E * exp2_fast(LOG2E * bf_hi(xw[e]));
            lam[e][0] = __uint_as_float(__float_as_uint(x0) & in); lam[e][1] = __uint_as_float(__float_as_uint(x1) & in);
            tot[0] += lam[e][0]; tot[1] += lam[e][1];
        }
        other[0] = __shfl_xor(tot[0], 32, 64); other[1] = __shfl_xor(tot[1], 32, 64);
        if (lane < 32) *reinterpret_cast<float2*>(&S.sums[wv][2 * p]) = make_float2(tot[0] + other[0], tot[1] + other[1]);
        __syncthreads();
        float off[2] = {0.f, 0.f}, all[2] = {0.f, 0.f};
#pragma unroll
        for (int z = 0; z < 16; ++z) {
            const float2 x = *reinterpret_cast<const float2*>(&S.sums[z][2 * p]);
            const uint32_t between = static_cast<uint32_t>((REV ? z - wv : wv - z) >> 31);
            off[0] += __uint_as_float(__float_as_uint(x.x) & between); off[1] += __uint_as_float(__float_as_uint(x.y) & between);
            all[0] += x.x; all[1] += x.y;
        }
        if (wv == 0) {
            if (lane < 32) *reinterpret_cast<float2*>(&S.total[2 * p]) = make_float2(all[0], all[1]);
            logd[0] += all[0]; logd[1] += all[1];
        }
        if (on) {
            if (REV ? half == 1 : half == 0) { off[0] += other[0]; off[1] += other[1]; }
#pragma unroll
            for (int z = 0; z < 8; ++z) {
                const int e = REV ? z : 7 - z;
                const uint32_t k2 = xk[e] & static_cast<uint32_t>((tk + e - live) >> 31);
                const HL y = hilo2k(bf_lo(k2) * exp2_fast(off[0]), bf_hi(k2) * exp2_fast(off[1]));
                const lds_t o = sb + (tk + e) * ROWL + 4 * p;
                lds_st<uint32_t>(o, y.h); lds_st<uint32_t>(o + PLANEL, y.l);
                off[0] += lam[e][0]; off[1] += lam[e][1];
            }
#pragma unroll
            for (int z = 0; z < 2; ++z)
                lds_st<u32x4>(sb + 2 * PLANEL + (vrow + 8 * z) * ROWL + 16 * vpc, u32x4{xv[z].x, xv[z].y, xv[z].z, xv[z].w} & static_cast<uint32_t>((vrow + 8 * z - live) >> 31));
        }
        __syncthreads();
        if (i + 1 < parts) fetch(REV ? part - 1 : part + 1);
        const f32x4 d = *reinterpret_cast<const f32x4*>(&S.total[16 * jt + 4 * g]);
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] *= exp2_fast(d[v]);
        // acc[v] = E[i = 16 it + l16][j = 16 jt + 4 g + v]
        lds_t k = sb + (8 * g + (l16 >> 2)) * ROWL + 8 * (l16 & 3);
        opaque(k);
        f32x4 lo = {0.f, 0.f, 0.f, 0.f};
        const lds_t kj = k + 32 * jt, vi = k + 2 * PLANEL + 32 * it;
#pragma unroll
        for (int s = 0; s < SUP / 32; ++s) {             // (all of them: without branches the reads run ahead)
            const bf16x8 v = ld_tr(vi + 32 * s * ROWL, ROWL);
            acc = mfma(ld_tr(kj + 32 * s * ROWL, ROWL), v, acc);
            lo = mfma(ld_tr(kj + PLANEL + 32 * s * ROWL, ROWL), v, lo);
        }
        acc += lo;
    }
    const size_t bq = static_cast<size_t>(bh) * a.NB + blk;
    *reinterpret_cast<f32x4*>(a.state + bq * (N * N) + (16 * it + l16) * N + 16 * jt + 4 * g) = acc;
    if (wv == 0 && lane < 32) *reinterpret_cast<float2*>(a.decay + bq * N + 2 * p) = make_float2(logd[0], logd[1]);
}

}  // namespace

int launch_wkv6_local(hipStream_t st, bool reverse, bool head_decay, int B, int T, int C, int H, int NB, int TB, const uint16_t* key, const uint16_t* val,
                      const uint16_t* w, float* state, float* decay, int* flags) {
    ArgsL a{T, C, H, NB, TB, key, val, w, state, decay, flags};
    const auto kernel = reverse ? (head_decay ? wkv6_local<true, true> : wkv6_local<true, false>) : (head_decay ? wkv6_local<false, true> : wkv6_local<false, false>);
    hipLaunchKernelGGL(kernel, dim3(B * H * NB), dim3(NTL), 0, st, a);
    return launch_status();
}

}  // namespace rwkv
