// fp32 products on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16): an fp32 value as three bf16 terms, x = h + m + l (rounded to
// nearest, every remainder exact), a product as the six that count, hh + hm + mh + mm + hl + lh; those left out are at most 2^-24 of it,
// 2^-27 in the root mean square.  Accumulation is fp32 either way.  All 24 bits from 2^-110 up to the largest fp32; what is smaller,
// a value (its last term falls among bf16's subnormals) or a product, is kept to about 2^-134.
//
// Why not v_mfma_f32_16x16x4_f32: it holds the vector unit.  Per SIMD, one wave issuing matrix and another vector instructions, cycles
// for 16 matrix and 64 vector ones: fp32 573 and 329 alone, 882 together; bf16 292 and 308 alone, 478 together.  16 elements of a
// contraction are four fp32 instructions (143 cycles, none left for anything else) or, two by two, three of these (55, of which the
// vector unit loses 30); 16 alone take four, two where one side is exact in bf16.  Splitting costs 5.5 vector instructions an element,
// 6.5 where infinite first terms have to be ruled out, once for all products that it enters.
//
// An infinity has a remainder that is no number: what it enters is NaN, where fp32 instructions would give an infinity or NaN.
#pragma once
#include "common.h"

namespace rwkv {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t lds_t;            // a byte address in the workgroup's LDS
template <class T> DEVINL T lds_ld(const lds_t a) { return *(const __attribute__((address_space(3))) T*)(a); }
template <class T> DEVINL void lds_st(const lds_t a, const T v) { *(__attribute__((address_space(3))) T*)(a) = v; }
DEVINL lds_t lds_of(const void* p) { return static_cast<lds_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)p)); }

// (an address behind an empty asm: an LDS offset beyond 64 KB does not fit an instruction, and the compiler would add it up again for
// every access instead of keeping a base)
DEVINL void opaque(lds_t& x) { asm volatile("" : "+v"(x)); }

DEVINL f32x4 mmb(const bf16x8& a, const bf16x8& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
DEVINL bf16x8 op2(const u32x2& a, const u32x2& b) { return __builtin_bit_cast(bf16x8, u32x4{a[0], a[1], b[0], b[1]}); }

// two values rounded to bf16; behind an empty asm, or the compiler converts once more to have them back as fp32
DEVINL uint32_t round2(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 p = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
    uint32_t r = __builtin_bit_cast(uint32_t, p);
    asm("" : "+v"(r));
    return r;
}
// The pair with an infinity replaced by the largest bf16 of its sign, in all of 16-bit integers: what is beyond 0x7f7f on the positive
// side, on the negative one what is beyond 0xff7f as unsigned numbers.  Two instructions a pair: B8 T1024 C4096, backward, fp32 mode
// 802 -> 826 us, bf16 613 -> 638 (in a form with a few spills); forward 376 -> 382 and 319 -> 327.  (Values held to that bound before they are rounded cost the
// backward registers: 796 -> 904 and 601 -> 641.  Looking for such values first and branching: 842 and 624.)  Not as inline assembly: a
// matrix instruction has to stay two wait states behind a vector instruction that writes its operand, and the compiler, which sees
// to that, does not look into assembly.
DEVINL uint32_t finite2(uint32_t r) {
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    const i16x2 p = __builtin_elementwise_min(__builtin_bit_cast(i16x2, r), i16x2{0x7f7f, 0x7f7f});
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, p), u16x2{0xff7f, 0xff7f}));
}
// four values, three terms.  A value beyond the largest bf16, (2 - 2^-7) 2^127, would round to an infinity, and its remainders were no
// numbers: its first term is that largest one and the others take the rest (below 2^120, so still exact).  BOUNDED: there is none.
struct B3 { u32x2 h, m, l; };
template <bool BOUNDED = false> DEVINL B3 split3(const f32x4& x) {
    B3 o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
        if constexpr (BOUNDED) o.h[i] = round2(a, b);
        else o.h[i] = finite2(round2(a, b));
        a -= bf_lo(o.h[i]); b -= bf_hi(o.h[i]);
        o.m[i] = round2(a, b);
        a -= bf_lo(o.m[i]); b -= bf_hi(o.m[i]);
        o.l[i] = round2(a, b);
    }
    return o;
}
// Contraction over 32: slots 0..3 of a lane from x, 4..7 from y
struct Op3 { bf16x8 h, m, l; };
DEVINL Op3 join(const B3& x, const B3& y) { return {op2(x.h, y.h), op2(x.m, y.m), op2(x.l, y.l)}; }
// Products of one size meet in one instruction, and the sum of the large ones is kept apart from the others until it is complete:
// eight products are added up before the rest of the sum, and what is small beside the largest of them loses bits.  Relative errors
// against 64 bits: 32 products of one size 2.9e-8, with half of them 2^-16 of the others 4.0e-8, onto a large sum 5.1e-8.
struct Sum2 { f32x4 hi, lo; };
constexpr Sum2 SUM0 = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
DEVINL f32x4 total(const Sum2& s) { return s.hi + s.lo; }
// (the sum is made before what follows: the compiler moves products that only a later phase takes behind the barrier between)
DEVINL void here(Sum2& s) { asm volatile("" : "+v"(s.hi), "+v"(s.lo)); }
DEVINL void add32(Sum2& s, const Op3& a, const Op3& b) {
    s.lo = mmb(a.l, b.h, s.lo);
    s.lo = mmb(a.h, b.l, s.lo);
    s.lo = mmb(a.m, b.m, s.lo);
    s.lo = mmb(a.m, b.h, s.lo);
    s.lo = mmb(a.h, b.m, s.lo);
    s.hi = mmb(a.h, b.h, s.hi);
}
// one side exact in bf16
DEVINL void add32(Sum2& s, const bf16x8& a, const Op3& b) { s.lo = mmb(a, b.m, mmb(a, b.l, s.lo)); s.hi = mmb(a, b.h, s.hi); }
// Contraction over 16, four elements a lane on either side: the halves of an instruction's 32 slots take different terms.
DEVINL void add16(Sum2& s, const B3& a, const B3& b) {
    const u32x2 z = {0u, 0u};
    s.lo = mmb(op2(a.l, a.h), op2(b.h, b.l), s.lo);
    s.lo = mmb(op2(a.m, z), op2(b.m, z), s.lo);
    s.lo = mmb(op2(a.h, a.m), op2(b.m, b.h), s.lo);
    s.hi = mmb(op2(a.h, z), op2(b.h, z), s.hi);
}
DEVINL void add16(Sum2& s, const B3& a, const u32x2& b) {
    s.lo = mmb(op2(a.l, a.m), op2(b, b), s.lo);
    s.hi = mmb(op2(a.h, u32x2{0u, 0u}), op2(b, b), s.hi);
}
DEVINL B3 as3(const B3& x) { return x; }
DEVINL B3 as3(const u32x2& x) { return {x, u32x2{0u, 0u}, u32x2{0u, 0u}}; }

// Planes of 64 channels x 16 tokens, [channel][token] bf16, one after the other for the terms.  A channel's four groups of four tokens
// are turned by the channel's number / 8, so that a wave's 8-byte pieces (lane = channel, or 16 channels by four groups) meet every
// bank once.
constexpr uint32_t TERM = 64 * 32, PLANE3 = 3 * TERM;
// piece of channel ch, tokens 4 tg + 0..3
DEVINL lds_t piece(int ch, int tg) { return static_cast<lds_t>(ch * 32 + 8 * (tg ^ ((ch >> 3) & 3))); }
DEVINL void put3(lds_t a, const B3& x) { lds_st<u32x2>(a, x.h); lds_st<u32x2>(a + TERM, x.m); lds_st<u32x2>(a + 2 * TERM, x.l); }
DEVINL B3 get3(lds_t a) { return {lds_ld<u32x2>(a), lds_ld<u32x2>(a + TERM), lds_ld<u32x2>(a + 2 * TERM)}; }
// Contraction over channels: lane <-> token l16, slots of block hb (32 channels) <-> channel 32 hb + 16 (e >> 2) + 4 g + (e & 3), i.e. as
// an accumulator holds them.  o = transposed(l16, g); 16 lanes read a 4 x 16 block, each ends up with a column.
DEVINL lds_t transposed(int l16, int g) { return static_cast<lds_t>((4 * g + (l16 >> 2)) * 32 + 8 * ((l16 & 3) ^ (g >> 1))); }
struct Tr { lds_t a, b; };           // the addresses of the two blocks of 16 channels (the second one's tokens are turned by two groups)
DEVINL Tr tr_bases(lds_t base, int l16, int g) { const lds_t o = transposed(l16, g); return {base + o, base + (o ^ 16u) + 512}; }
DEVINL bf16x8 ld_tr16(const Tr& o, uint32_t plane, int hb) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef v4s __attribute__((address_space(3))) * ptr;
    const v4s x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(o.a + plane + 1024 * hb)), y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(o.b + plane + 1024 * hb));
    return op2(__builtin_bit_cast(u32x2, x), __builtin_bit_cast(u32x2, y));
}
DEVINL Op3 get3_tr(uint32_t plane, const Tr& o, int hb) { return {ld_tr16(o, plane, hb), ld_tr16(o, plane + TERM, hb), ld_tr16(o, plane + 2 * TERM, hb)}; }

// Two planes (x, y) whose products share instructions, which are also read over channels one by one: a channel's row is 32 bytes of x
// and 32 of y, 32 bytes more behind every four channels, and its pieces are turned by the channel's number, bits reversed.  So the pieces
// that half a wave reads or writes meet every bank once: of four channels by four groups, two groups (transposing), of sixteen by two
// (rows), of 32 channels (P waves).  (x and y in turn, 16 bytes a piece: one instruction reads both, but the transposing reads use half of
// the banks: in rwkv7c_bwd 38 % of the LDS's active time were conflicts, 23 % so, and the time goes from 599 to 591 us.)
constexpr uint32_t TWIN = 64 * 64 + 16 * 32, TWIN3 = 3 * TWIN, TWIN_ROWS = 1152;      // a term; 16 channels on
DEVINL lds_t twin(int ch, int tg) { return static_cast<lds_t>(64 * ch + 32 * (ch >> 2) + 8 * (tg ^ ((ch & 1) << 1 | (ch >> 1 & 1)))); }
DEVINL void put_twin(lds_t a, const B3& x, const B3& y) {
    lds_st<u32x2>(a, x.h); lds_st<u32x2>(a + 32, y.h);
    lds_st<u32x2>(a + TWIN, x.m); lds_st<u32x2>(a + TWIN + 32, y.m);
    lds_st<u32x2>(a + 2 * TWIN, x.l); lds_st<u32x2>(a + 2 * TWIN + 32, y.l);
}
DEVINL Op3 get_twin(lds_t a) {
    return {op2(lds_ld<u32x2>(a), lds_ld<u32x2>(a + 32)), op2(lds_ld<u32x2>(a + TWIN), lds_ld<u32x2>(a + TWIN + 32)), op2(lds_ld<u32x2>(a + 2 * TWIN), lds_ld<u32x2>(a + 2 * TWIN + 32))};
}
// one of the two over channels, as get3_tr (y: 32 bytes on)
DEVINL lds_t tr_twin(lds_t base, int l16, int g) { return base + twin(4 * g + (l16 >> 2), l16 & 3); }
DEVINL bf16x8 ld_tr16_twin(lds_t o, uint32_t plane, int hb) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef v4s __attribute__((address_space(3))) * ptr;
    const v4s x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(o + plane + 2 * TWIN_ROWS * hb)), y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(o + plane + 2 * TWIN_ROWS * hb + TWIN_ROWS));
    return op2(__builtin_bit_cast(u32x2, x), __builtin_bit_cast(u32x2, y));
}
DEVINL Op3 get3_tr_twin(uint32_t plane, lds_t o, int hb) { return {ld_tr16_twin(o, plane, hb), ld_tr16_twin(o, plane + TWIN, hb), ld_tr16_twin(o, plane + 2 * TWIN, hb)}; }

// Two tiles whose products share instructions, interleaved by pieces: 16 bytes are a side of one instruction.  (Held apart,
// each would be read by itself and its halves moved together.)  Of a tile a lane holds row l16, columns 4 g + 0..3, as a side of a
// contraction over the columns takes them.
constexpr uint32_t TTERM2 = 1024, TPAIR3 = 3 * TTERM2;
DEVINL lds_t piece2(int row, int piece) { return static_cast<lds_t>(row * 64 + 16 * (piece ^ ((row >> 2) & 3))); }      // (a channel's 16 bytes of four tokens lie so as well)
template <uint32_t STRIDE> DEVINL void put_half(lds_t a, const B3& x) { lds_st<u32x2>(a, x.h); lds_st<u32x2>(a + STRIDE, x.m); lds_st<u32x2>(a + 2 * STRIDE, x.l); }
template <uint32_t STRIDE> DEVINL B3 get_half(lds_t a) { return {lds_ld<u32x2>(a), lds_ld<u32x2>(a + STRIDE), lds_ld<u32x2>(a + 2 * STRIDE)}; }
template <uint32_t STRIDE> DEVINL Op3 get_pair(lds_t a) {
    return {__builtin_bit_cast(bf16x8, lds_ld<u32x4>(a)), __builtin_bit_cast(bf16x8, lds_ld<u32x4>(a + STRIDE)), __builtin_bit_cast(bf16x8, lds_ld<u32x4>(a + 2 * STRIDE))};
}

}  // namespace
}  // namespace rwkv
