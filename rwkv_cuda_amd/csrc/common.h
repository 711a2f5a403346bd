// Shared device helpers and host-side argument checks for librwkv_hip.so (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <utility>

#include "rwkv_hip.h"

#define DEVINL __device__ __forceinline__

namespace rwkv {

// ----------------------------------------------------------------------------- bf16 <-> f32
DEVINL float bf2f(uint16_t x) { return __uint_as_float(static_cast<uint32_t>(x) << 16); }
DEVINL float bf_lo(uint32_t x) { return __uint_as_float(x << 16); }          // element 0 of a packed pair
DEVINL float bf_hi(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }  // element 1 of a packed pair

// fp32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950; NaN stays NaN)
DEVINL uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }
DEVINL uint32_t pack_bf2(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const bf16x2_t p = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
    return __builtin_bit_cast(uint32_t, p);
}

DEVINL void unpack8(const uint4& q, float (&f)[8]) {
    f[0] = bf_lo(q.x); f[1] = bf_hi(q.x); f[2] = bf_lo(q.y); f[3] = bf_hi(q.y);
    f[4] = bf_lo(q.z); f[5] = bf_hi(q.z); f[6] = bf_lo(q.w); f[7] = bf_hi(q.w);
}
DEVINL uint4 pack8(const float (&f)[8]) {
    uint4 q;
    q.x = pack_bf2(f[0], f[1]); q.y = pack_bf2(f[2], f[3]);
    q.z = pack_bf2(f[4], f[5]); q.w = pack_bf2(f[6], f[7]);
    return q;
}

// ----------------------------------------------------------------------------- row broadcast
// A wave64 is four DPP rows of 16 lanes.  bc<J>(x) is x of lane (row*16 + J): with a vector
// laid out as x_lane = vec[base + (lane & 15)] this gives vec[base + J] in every lane without
// an LDS read or an SGPR.  The fused forms below put the broadcast inside the VALU op
// (v_fmac_f32_dpp / v_mul_f32_dpp row_newbcast), so a broadcast operand costs nothing.
// The DPP source operand must not have been written by the one or two VALU instructions
// just before (gfx9 DPP read-after-VALU-write hazard); callers only feed it values that come
// straight from LDS or that are loop invariant.
template <int J> DEVINL void fmac_bc(float& acc, float row_vec, float s) {   // acc += row_vec[J] * s
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(acc) : "v"(row_vec), "v"(s), "n"(J));
}
template <int J> DEVINL void mul_bc(float& s, float row_vec) {               // s *= row_vec[J]
    asm("v_mul_f32_dpp %0, %1, %0 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
        : "+v"(s) : "v"(row_vec), "n"(J));
}
// The sums of a triangular solve by such broadcasts: SOLVE_ROWS m[s] += x[t][lane s] m[t] for t from 15 down and s < t, SOLVE_COLS for t
// from 0 up and s > t.  x[t] comes from wherever the caller's code left it, so all of it is one statement behind its own wait states:
// between single ones the compiler could copy an x[t] and, as it does not look into assembly, leave out the wait.
#define RWKV_BC(t, x, s) "v_fmac_f32_dpp %" #s ", %" #x ", %" #t " row_newbcast:" #s " row_mask:0xf bank_mask:0xf\n\t"
#define RWKV_DOWN1(t, x) RWKV_BC(t, x, 0)
#define RWKV_DOWN2(t, x) RWKV_BC(t, x, 1) RWKV_DOWN1(t, x)
#define RWKV_DOWN3(t, x) RWKV_BC(t, x, 2) RWKV_DOWN2(t, x)
#define RWKV_DOWN4(t, x) RWKV_BC(t, x, 3) RWKV_DOWN3(t, x)
#define RWKV_DOWN5(t, x) RWKV_BC(t, x, 4) RWKV_DOWN4(t, x)
#define RWKV_DOWN6(t, x) RWKV_BC(t, x, 5) RWKV_DOWN5(t, x)
#define RWKV_DOWN7(t, x) RWKV_BC(t, x, 6) RWKV_DOWN6(t, x)
#define RWKV_DOWN8(t, x) RWKV_BC(t, x, 7) RWKV_DOWN7(t, x)
#define RWKV_DOWN9(t, x) RWKV_BC(t, x, 8) RWKV_DOWN8(t, x)
#define RWKV_DOWN10(t, x) RWKV_BC(t, x, 9) RWKV_DOWN9(t, x)
#define RWKV_DOWN11(t, x) RWKV_BC(t, x, 10) RWKV_DOWN10(t, x)
#define RWKV_DOWN12(t, x) RWKV_BC(t, x, 11) RWKV_DOWN11(t, x)
#define RWKV_DOWN13(t, x) RWKV_BC(t, x, 12) RWKV_DOWN12(t, x)
#define RWKV_DOWN14(t, x) RWKV_BC(t, x, 13) RWKV_DOWN13(t, x)
#define RWKV_DOWN15(t, x) RWKV_BC(t, x, 14) RWKV_DOWN14(t, x)
#define RWKV_UP15(t, x) RWKV_BC(t, x, 15)
#define RWKV_UP14(t, x) RWKV_BC(t, x, 14) RWKV_UP15(t, x)
#define RWKV_UP13(t, x) RWKV_BC(t, x, 13) RWKV_UP14(t, x)
#define RWKV_UP12(t, x) RWKV_BC(t, x, 12) RWKV_UP13(t, x)
#define RWKV_UP11(t, x) RWKV_BC(t, x, 11) RWKV_UP12(t, x)
#define RWKV_UP10(t, x) RWKV_BC(t, x, 10) RWKV_UP11(t, x)
#define RWKV_UP9(t, x) RWKV_BC(t, x, 9) RWKV_UP10(t, x)
#define RWKV_UP8(t, x) RWKV_BC(t, x, 8) RWKV_UP9(t, x)
#define RWKV_UP7(t, x) RWKV_BC(t, x, 7) RWKV_UP8(t, x)
#define RWKV_UP6(t, x) RWKV_BC(t, x, 6) RWKV_UP7(t, x)
#define RWKV_UP5(t, x) RWKV_BC(t, x, 5) RWKV_UP6(t, x)
#define RWKV_UP4(t, x) RWKV_BC(t, x, 4) RWKV_UP5(t, x)
#define RWKV_UP3(t, x) RWKV_BC(t, x, 3) RWKV_UP4(t, x)
#define RWKV_UP2(t, x) RWKV_BC(t, x, 2) RWKV_UP3(t, x)
#define RWKV_UP1(t, x) RWKV_BC(t, x, 1) RWKV_UP2(t, x)
#define RWKV_SOLVE_OPERANDS \
    : "+&v"(m[0]), "+&v"(m[1]), "+&v"(m[2]), "+&v"(m[3]), "+&v"(m[4]), "+&v"(m[5]), "+&v"(m[6]), "+&v"(m[7]), \
      "+&v"(m[8]), "+&v"(m[9]), "+&v"(m[10]), "+&v"(m[11]), "+&v"(m[12]), "+&v"(m[13]), "+&v"(m[14]), "+&v"(m[15]) \
    : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), \
      "v"(x[8]), "v"(x[9]), "v"(x[10]), "v"(x[11]), "v"(x[12]), "v"(x[13]), "v"(x[14]), "v"(x[15])
template <bool ROWS> DEVINL void solve_bc(float (&m)[16], const float (&x)[16]) {      // operands 0..15 are m, 16..31 x
    if constexpr (ROWS)
        asm("s_nop 1\n\t"
            RWKV_DOWN15(15, 31) RWKV_DOWN14(14, 30) RWKV_DOWN13(13, 29) RWKV_DOWN12(12, 28) RWKV_DOWN11(11, 27)
            RWKV_DOWN10(10, 26) RWKV_DOWN9(9, 25) RWKV_DOWN8(8, 24) RWKV_DOWN7(7, 23) RWKV_DOWN6(6, 22)
            RWKV_DOWN5(5, 21) RWKV_DOWN4(4, 20) RWKV_DOWN3(3, 19) RWKV_DOWN2(2, 18) RWKV_DOWN1(1, 17)
            RWKV_SOLVE_OPERANDS);
    else
        asm("s_nop 1\n\t"
            RWKV_UP1(0, 16) RWKV_UP2(1, 17) RWKV_UP3(2, 18) RWKV_UP4(3, 19) RWKV_UP5(4, 20)
            RWKV_UP6(5, 21) RWKV_UP7(6, 22) RWKV_UP8(7, 23) RWKV_UP9(8, 24) RWKV_UP10(9, 25)
            RWKV_UP11(10, 26) RWKV_UP12(11, 27) RWKV_UP13(12, 28) RWKV_UP14(13, 29) RWKV_UP15(14, 30)
            RWKV_SOLVE_OPERANDS);
}
template <int J> DEVINL float bc(float row_vec) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, row_vec),
                                                                0x150 + J, 0xf, 0xf, true));
}

template <typename F, int... I> DEVINL void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> DEVINL void static_for(F&& f) {
    static_for_impl(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

// sum over a group of 2^k consecutive lanes (k <= 6); result valid in every lane of the group
template <int WIDTH> DEVINL float group_sum(float x) {
#pragma unroll
    for (int m = WIDTH / 2; m >= 1; m >>= 1) x += __shfl_xor(x, m, 64);
    return x;
}

// sum over the four 16-lane rows of a wave (lanes l, l^16, l^32, l^48); result in all four.
// Two register-swap steps: permlane16_swap exchanges odd rows of one copy with even rows of
// the other, permlane32_swap exchanges the wave halves; neither touches LDS.  The s_nop
// covers the wait states a swap needs after a VALU write of its operands.
DEVINL float allreduce_rows(float x) {
#if RWKV_ROWSUM_SHFL
    x += __shfl_xor(x, 16, 64);
    x += __shfl_xor(x, 32, 64);
    return x;
#else
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    float s = a + b;
    a = s; b = s;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return a + b;
#endif
}

// The same two swaps applied to distinct values do more work per instruction.  permlane16_swap(a, b) leaves
// a = [a0, b0, a2, b2] and b = [a1, b1, a3, b3] (by row), permlane32_swap(s, t) leaves s = [s0, s1, t0, t1] and
// t = [s2, s3, t2, t3].

// Row sums of four values in three swaps: row 0 of the result holds sum(a), row 1 sum(b), row 2 sum(c), row 3 sum(d).
DEVINL float reduce4_rows(float a, float b, float c, float d) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1"
                 : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
    float s = a + b, t = c + d;                   // [a01, b01, a23, b23], [c01, d01, c23, d23]
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(s), "+v"(t));
    return s + t;
}

// Row sums of two values, each result in all four rows, in three swaps instead of four.
DEVINL void allreduce2_rows(float& x, float& y) {
    float a = x, b = y;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    float s = a + b;                              // [x01, y01, x23, y23]
    float t = s;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(s), "+v"(t));
    float u = s + t;                              // [X, Y, X, Y]
    float w = u;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(u), "+v"(w));
    x = u; y = w;                                 // [X, X, X, X], [Y, Y, Y, Y]
}

// ----------------------------------------------------------------------------- wkv5: decays that are too fast for chunks
// wkv5's chunked kernels carry powers e^{l d} of a channel's log decay l = -exp(w) over a few tokens, in both directions.  A head
// with one channel beyond what they carry (fp32 wkv5c_*: l < -17, where the powers of half a chunk still stay inside fp32; bf16
// wkv5b_*: l < -9, half a chunk of twice the length) runs step by step instead (wkv5_steps_*, wkv56.hip).  A decay that is no
// number counts as one of these: the steps hand it on as the operator does.  Chunked and step kernels decide by the same test,
// for the channels of the head from c0 on.
constexpr float W_STEPS_F32 = 2.8332133f, W_STEPS_BF16 = 2.1875f;      // ln 17; e^2.1875 = 8.91, the last bfloat16 below ln 9
template <bool F32, int HN> DEVINL bool steps_head(const void* w, const void* w2, const int c0) {
    bool on = false;
#pragma unroll
    for (int z = 0; z < HN / 64; ++z) {
        const int c = c0 + 64 * z + (threadIdx.x & 63);
        if constexpr (F32) on |= !(static_cast<const float*>(w)[c] <= W_STEPS_F32);
        else on |= !(bf2f(static_cast<const uint16_t*>(w)[c]) <= W_STEPS_BF16);
        if (F32 && w2 != nullptr) on |= !(static_cast<const float*>(w2)[c] <= W_STEPS_F32);
    }
    return __ballot(on) != 0ull;
}
// bf16, heads of 64: whether any channel of the layer decays faster than the mid-point factors of the one-sweep kernels
// (wkv6_fwd_f.hip, wkv6_bwd_f.hip) carry (16 tokens by more than e^-60: w > 1.32; the threshold is the bfloat16 below), or is no
// number.  One such channel moves the whole layer to wkv5_bf.hip: redoing the one head after the others would cost the time of the
// longest sequence once more (B8 T4096 C2048, forward + backward: 0.54 ms in one sweep; there 0.69 ms with a channel at w = 1.5 or
// 2.15; 3.1 ms with the one head step by step, as a head beyond W_STEPS_BF16 still is).  Every wave looks at every channel (C is a multiple of 64), so
// all come to the same answer.
DEVINL bool strong_decay(const float w) { return !(w <= 1.3125f); }
DEVINL bool strong_layer(const uint16_t* w, const int C, const int lane) {
    bool strong = false;
    for (int c = lane * 8; c < C; c += 512) {
        float f[8];
        unpack8(*reinterpret_cast<const uint4*>(w + c), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) strong |= strong_decay(f[e]);
    }
    return __ballot(strong) != 0ull;
}

// ----------------------------------------------------------------------------- host checks
extern thread_local int g_last_hip_error;

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// need_align: the kernels that will run use 16-byte loads and stores (those for other head sizes than 64 do not)
inline int check_ptrs(std::initializer_list<const void*> ps, bool need_align = true) {
    for (const void* p : ps) if (p == nullptr) return RWKV_ERR_NULL;
    if (need_align) for (const void* p : ps) if (!aligned16(p)) return RWKV_ERR_ALIGN;
    return RWKV_OK;
}

inline int launch_status() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { g_last_hip_error = static_cast<int>(e); return RWKV_ERR_LAUNCH; }
    return RWKV_OK;
}

// ----------------------------------------------------------------------------- internal launchers
// wkv6_chunk.hip: chunked MFMA kernels.  wmode: 1 = fp32 ew [B,T,C], 2 = raw bf16 w.
int launch_wkv6_fwd_chunk(hipStream_t st, int wmode, int B, int T, int C, int H, const uint16_t* r,
                          const uint16_t* k, const uint16_t* v, const void* w, const uint16_t* u,
                          const uint16_t* s0, uint16_t* y, char* saved = nullptr, const int* only_flagged = nullptr);
// wkv6_fwd_f.hip: the forward that goes with wkv6_bwd_f.hip (raw bf16 decay, head size 64): y and the state entering
// every second chunk; flags [B*H][8] names the (batch, head) pairs that have to be redone by the kernel above
// NB > 1: the sequences in NB blocks of TB tokens, one workgroup per (batch, head, block): local states, a scan, the outputs
// (blk_state, s32: [B*H*NB][64][64] floats each, blk_decay: [B*H*NB][64])
int launch_wkv6_fwd_fused(hipStream_t st, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k, const uint16_t* v,
                          const uint16_t* w, const uint16_t* u, const uint16_t* s0, uint16_t* y, char* saved, int* flags,
                          int NB = 1, int TB = 0, float* blk_state = nullptr, float* blk_decay = nullptr, float* s32 = nullptr,
                          float* decay_out = nullptr);
// wkv6_local.hip: the first of these, for either direction (backward: key = r, val = gy); flags are cleared
int launch_wkv6_local(hipStream_t st, bool reverse, bool head_decay, int B, int T, int C, int H, int NB, int TB, const uint16_t* key, const uint16_t* val,
                      const uint16_t* w, float* state, float* decay, int* flags);
// As many blocks as this at most: what enters a block is added up by the kernel that starts from there, while its loads are under way.  B1 H32
// T3001, 8 blocks, forward + backward 109.5 us with wkv6_scan between (4.3 us each way), 106.3 without; B1 H8 T2000, 16 blocks, forward
// 30.7 and 30.1; a step of the sum takes about 0.7 us.
constexpr int SCAN_BLOCKS = 16;
int launch_wkv6_scan_reverse(hipStream_t st, int BH, int NB, const float* local, const float* logdec, float* out);
int launch_wkv6_bwd_a_chunk(hipStream_t st, int wmode, int B, int T, int C, int H, const uint16_t* r,
                            const uint16_t* k, const uint16_t* v, const void* w, const uint16_t* u,
                            const uint16_t* s0, const uint16_t* gy, uint16_t* gr, uint16_t* gu, float* rdr,
                            const int* only_flagged = nullptr, const float* gu_parts = nullptr, int gu_blocks = 0);
int launch_wkv6_bwd_b_chunk(hipStream_t st, int wmode, int B, int T, int C, int H, const uint16_t* r,
                            const uint16_t* k, const uint16_t* v, const void* w, const uint16_t* u,
                            const uint16_t* s0, const uint16_t* gy, uint16_t* gk, uint16_t* gv, uint16_t* gw,
                            uint16_t* gs, const float* rdr, const int* only_flagged = nullptr,
                            const uint16_t* sum_in = nullptr, uint16_t* sum_out = nullptr);
// wkv6_bwd_f.hip: the whole backward in one reverse sweep from the states the forward saved (raw bf16 decay);
// flags [B*H][8] names the (batch, head) pairs that have to be redone by the two sweeps above
int launch_wkv6_bwd_fused(hipStream_t st, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k, const uint16_t* v,
                          const uint16_t* w, const uint16_t* u, const uint16_t* gy, uint16_t* gr, uint16_t* gk, uint16_t* gv,
                          uint16_t* gw, uint16_t* gu, uint16_t* gs, const char* saved, int* flags,
                          int NB = 1, int TB = 0, float* blk_ds = nullptr, float* blk_decay = nullptr, float* ds32 = nullptr,
                          float* gu32 = nullptr, uint16_t* gwp = nullptr, float* gw32 = nullptr);
// gwp != nullptr: wkv5 (w is the raw decay per channel [H][64]; its gradient per batch row goes to gwp [B][C], gw is not written)
// wkv5 with heads of 128 channels as four heads of 64 (see ArgsB in wkv6_chunk.h): one launch of each kernel per value
// of `cross`.  Forward and first sweep: the first launch (cross = 0) leaves fp32 terms, the second adds them to its own
// and writes the bf16 outputs.  Second sweep: both launches leave fp32 terms (its waves have no registers to spare for
// the first launch's terms), which the caller adds.
int launch_wkv5_fwd_split(hipStream_t st, int cross, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k,
                          const uint16_t* v, const float* eew, const uint16_t* u, float* y32, uint16_t* y);
int launch_wkv5_bwd_a_split(hipStream_t st, int cross, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k,
                            const uint16_t* v, const float* ew, const uint16_t* u, const uint16_t* gy, float* gr32, float* gu32,
                            uint16_t* gr, uint16_t* gu, float* rdr);
int launch_wkv5_bwd_b_split(hipStream_t st, int cross, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k,
                            const uint16_t* v, const float* ew, const uint16_t* u, const uint16_t* gy, float* gk32, float* gv32,
                            float* gw32, const float* rdr);
// wkv56.hip: the heads of an fp32 wkv5 (wkv5a: w2, u2 not null) layer of 64-channel heads that the chunked kernels leave out; gw, gu,
// gw2, gu2: per-batch rows [B][C]; flags (may be null): a word per (batch, head) that says so instead of the decays and marks
int launch_wkv5f32_steps_fwd(hipStream_t st, int B, int T, int H, const float* r, const float* k, const float* v, const float* w,
                             const float* u, const float* w2, const float* u2, float* y, const int* flags = nullptr);
int launch_wkv5f32_steps_bwd(hipStream_t st, int B, int T, int H, const float* r, const float* k, const float* v, const float* w,
                             const float* u, const float* w2, const float* u2, const float* gy, float* gr, float* gk, float* gv,
                             float* gw, float* gu, float* gw2, float* gu2, const int* flags = nullptr);

// wkv5_bf.hip: wkv5, bf16, heads of 128 or 64 channels, whole heads; w raw.  Size 64: only layers with a
// strong decay (strong_layer), the others belong to the one-sweep kernels above and the launch returns at once.
// Heads that run step by step (steps_head) are left out.  saved (may be null in the forward):
// the states for the backward; gw, gu: per-batch rows [B][C].
constexpr int WKV5B_MAX_C = 1 << 24;           // byte offsets within 32 rows are 32-bit
// ws (may be null: whole sequences): wkv5b_blocks_bytes, 16-byte aligned, for few sequences in blocks of time (heads of 128)
size_t wkv5b_saved_bytes(int B, int T, int C, int H);
size_t wkv5b_blocks_bytes(int B, int T, int C, int H, bool bwd);
int launch_wkv5b_fwd(hipStream_t st, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k, const uint16_t* v, const uint16_t* w,
                     const uint16_t* u, uint16_t* y, float* decay, float* saved, void* ws = nullptr);
int launch_wkv5b_bwd(hipStream_t st, int B, int T, int C, int H, const uint16_t* r, const uint16_t* k, const uint16_t* v, const uint16_t* w,
                     const uint16_t* u, const uint16_t* gy, uint16_t* gr, uint16_t* gk, uint16_t* gv, uint16_t* gw, uint16_t* gu,
                     const float* saved, void* ws = nullptr);

// rwkv7_chunk.hip: chunked rwkv7 kernels (r..b, y, dy, dr..db are bf16 or, with f32, float); s0, sT, dsT, ds0 may be null.  ws (may be
// null: whole sequences): rwkv7c_workspace_bytes, 16-byte aligned, for few sequences in blocks of time
size_t rwkv7c_workspace_bytes(int B, int T, int H, bool bwd);
int launch7c_fwd(hipStream_t st, bool f32, int B, int T, int H, const float* s0, const void* r, const void* w, const void* k,
                 const void* v, const void* a, const void* b, void* y, float* sT, float* s, float* sa, void* ws = nullptr);
int launch7c_bwd(hipStream_t st, bool f32, int B, int T, int H, const void* r, const void* w, const void* k, const void* v,
                 const void* a, const void* b, const void* dy, const float* dsT, const float* s, const float* sa,
                 float* ds0, void* dr, void* dw, void* dk, void* dv, void* da, void* db, void* ws = nullptr);

}  // namespace rwkv
