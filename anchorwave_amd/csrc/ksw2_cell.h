// ksw2_cell.h -- the two-piece-affine cell on packed 16-bit halves, shared by
// the kernels that work in the exactness domain (match 0, mismatch <= 0,
// every int8 intermediate of the reference in range).
//
// A register holds two cells, one in each half.  x and v come from the cell
// above, u and y from the cell to the left (x2, y2: the second gap piece):
//   z = max(s, a, b, a2, b2), a = x + v, b = y + u, a2 = x2 + v, b2 = y2 + u
//   u' = z - v, v' = z - u, x' = max(a - z + q, 0) - (q + e), y' likewise
// (minimap2/ksw2_extd2_sse.c:43-71, 237-331).  Everything is negated, so the
// maximum is a minimum of non-negative halves: in this domain every
// candidate is <= 0.  Two forms:
//
//  * DirCell, for direction bytes: values scaled by 8 under a 3-bit tag, so
//    the minimum also gives the index the reference's strict '>' chain (left
//    alignment: tags k) or '>=' chain (right alignment: tags 7-k) picks.
//    x and y are stored as -8(x + G1) - bias + tag (bias 0 left, 8 right):
//    the sign of the value before its clamp is the continuation flag.  v and
//    u are stored as -8v + p with p = 8 G1 + bias, which makes x + v and
//    y + u the tagged candidates with no further constant; the second
//    piece's candidates take one constant each.
//  * RawCell, for scores and Singletrack tracks: unscaled, no tags, no flags.
//
// What bounds it: VALU issue.  On gfx950 a packed 16-bit operation, a
// three-input bit operation, a permute and a three-input packed minimum each
// hold the SIMD for about 4.2 cycles when several waves share it, and 4.9 for
// a wave alone (measured in loops of one instruction, and of this cell), so
// what counts is the number of instructions.  The five-way minimum is two
// v_pk_minimum3_f16 instead of four v_pk_min_i16: halves in [0, 0x7bff] order
// the same as floats and as integers, subnormals included.  A row of two
// cells takes 27.5 instructions with its direction bytes and 19 without
// (35.5 and 26 in the form it replaced); eight rows of it with their
// direction store ran 1,041 cycles a step on four waves per SIMD against
// 1,377, and 1,225 against 1,943 on one.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ksw2_common.h"

namespace kswhip {
namespace cell {

typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned short v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t splat(int x) { return (uint32_t)(x & 0xffff) * 0x10001u; }
__device__ __forceinline__ int lo16(uint32_t x) { return (int)(int16_t)(x & 0xffffu); }
__device__ __forceinline__ int hi16(uint32_t x) { return (int)x >> 16; }

__device__ __forceinline__ uint32_t add2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2u, a) + __builtin_bit_cast(v2u, b));
}
__device__ __forceinline__ uint32_t sub2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2u, a) - __builtin_bit_cast(v2u, b));
}
__device__ __forceinline__ uint32_t min2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t,
                              __builtin_elementwise_min(__builtin_bit_cast(v2s, a), __builtin_bit_cast(v2s, b)));
}
__device__ __forceinline__ uint32_t max2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t,
                              __builtin_elementwise_max(__builtin_bit_cast(v2s, a), __builtin_bit_cast(v2s, b)));
}
// All ones in the halves that are negative.
__device__ __forceinline__ uint32_t sign2(uint32_t a)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2s, a) >> (v2s){15, 15});
}
// The low (high) half of a, signed, plus b.
__device__ __forceinline__ int add_lo(uint32_t a, int b) { return __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, a), (v2s){1, 0}, b, false); }
__device__ __forceinline__ int add_hi(uint32_t a, int b) { return __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, a), (v2s){0, 1}, b, false); }
// Smallest of three, per half; halves in [0, 0x7bff].
__device__ __forceinline__ uint32_t min3(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    asm("v_pk_minimum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// (a & m) | (b & ~m)
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t a, uint32_t b) { return __builtin_amdgcn_bitop3_b32(m, a, b, 0xca); }
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel)
{
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// Lane k takes lane k+1's value (lane 63 `old`), lane k takes lane k-1's
// (lane 0 `old`), lane k takes lane k-1's (lane 0 lane 63's).
__device__ __forceinline__ uint32_t dpp_shl1(uint32_t old, uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, 0x130, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t dpp_shr1(uint32_t old, uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, 0x138, 0xF, 0xF, false);
}
// Lane k takes lane k-1's value (lane 0 zero).
__device__ __forceinline__ uint32_t dpp_shr1_0(uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)src, 0x138, 0xF, 0xF, true);
}
// Lane k takes lane k+7's value where both are in a row of 16 lanes.
__device__ __forceinline__ uint32_t dpp_row_shl7(uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)src, 0x107, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t dpp_ror1(uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)src, 0x13C, 0xF, 0xF, false);
}

// State of two cells: x, x2, v go down (from the cells above to those
// below), u, y, y2 go right.
struct Down {
    uint32_t x, x2, v;
};
struct Right {
    uint32_t u, y, y2;
};

// Two cells' direction byte before packing: tags in the low bits of z, flags
// in bits 11-14 of f, one set in each half.
struct DirWord {
    uint32_t z, f;
};

template <bool RIGHT>
struct DirCell {
    static constexpr int kScale = 8;
    static constexpr int bias = RIGHT ? 8 : 0;
    static constexpr int tS = RIGHT ? 7 : 0;
    uint32_t cA2, cB2, zc, e1, e2, lA, lB, lA2, lB2;
    uint32_t mA, mB, mA2;  // flag bits of a and b; the bits of f taken from a2 rather than b2
    int p, sm, sx;         // v and u bias; score candidates of a match and a mismatch

    // A transposed pair (the reference's query in the rows, its target swept)
    // has above and left exchanged: its a and a2 are the reference's b and b2.
    // They take those candidates' tags and flag bits, which keeps the
    // reference's tie order and byte.
    __device__ __forceinline__ DirCell(const KswScore &sc, bool transposed)
    {
        const int t1 = RIGHT ? 6 : 1, t2 = RIGHT ? 5 : 2, t3 = RIGHT ? 4 : 3, t4 = RIGHT ? 3 : 4;
        const int tA = transposed ? t2 : t1, tB = transposed ? t1 : t2;
        const int tA2 = transposed ? t4 : t3, tB2 = transposed ? t3 : t4;
        // The reference's byte has a's flag in bit 3, b 4, a2 5, b2 6; f holds
        // bit k at k + 8.  |values before their clamp| < 2048, so bits 11-15
        // of one are all its sign.  The second-piece state whose flag goes to
        // bit 13 is biased by 0x4000: bits 11-13 are still its flag, bit 15 is
        // 0, and it gives the bits that no flag takes.
        const int bA2 = transposed ? 0 : 0x4000, bB2 = transposed ? 0x4000 : 0;
        const int d = 8 * (sc.G2 - sc.G1);
        p = 8 * sc.G1 + bias;
        cA2 = splat(d - bA2), cB2 = splat(d - bB2);
        zc = splat(2 * p);
        e1 = splat(-8 * sc.q - bias), e2 = splat(d - 8 * sc.q2 - bias);
        lA = splat(tA - bias), lB = splat(tB - bias);
        lA2 = splat(tA2 - bias + bA2), lB2 = splat(tB2 - bias + bB2);
        mA = transposed ? 0x10001000u : 0x08000800u, mB = transposed ? 0x08000800u : 0x10001000u;
        mA2 = transposed ? 0x40004000u : 0xbfffbfffu;
        sm = -8 * sc.mch + tS, sx = -8 * sc.mis + tS;
    }
    // x, x2, y, y2 of a boundary (no gap open), in both halves
    __device__ __forceinline__ uint32_t x0() const { return lA; }
    __device__ __forceinline__ uint32_t x20() const { return lA2; }
    __device__ __forceinline__ uint32_t y0() const { return lB; }
    __device__ __forceinline__ uint32_t y20() const { return lB2; }
    // one half of v or u for the difference w
    __device__ __forceinline__ int diff(int w) const { return p - 8 * w; }

    // STALE: some inputs were left by earlier anti-diagonals, outside a band;
    // their candidates may be positive (a negative half), and the score is
    // capped at the match score.
    template <bool STALE = false> __device__ __forceinline__ DirWord step(uint32_t s, Down &d, Right &r) const
    {
        const uint32_t a = add2(d.x, d.v), b = add2(r.y, r.u);
        const uint32_t xv2 = add2(d.x2, d.v), yu2 = add2(r.y2, r.u);
        const uint32_t a2 = add2(xv2, cA2), b2 = add2(yu2, cB2);
        const uint32_t z = STALE ? min2(min2(min2(b, b2), s), min2(a, a2)) : min3(min3(s, a, b), a2, b2);
        const uint32_t z8 = STALE ? max2(z & 0xfff8fff8u, 0u) : z & 0xfff8fff8u;
        const uint32_t w = add2(z8, zc), m1 = sub2(e1, z8), m2 = sub2(e2, z8);
        const uint32_t ta = add2(a, m1), tb = add2(b, m1), ta2 = add2(xv2, m2), tb2 = add2(yu2, m2);
        const uint32_t un = sub2(w, d.v);
        d.v = sub2(w, r.u), r.u = un;
        d.x = min2(ta, lA), r.y = min2(tb, lB), d.x2 = min2(ta2, lA2), r.y2 = min2(tb2, lB2);
        DirWord o;
        o.z = z, o.f = bfi(mA, ta, bfi(mB, tb, bfi(mA2, ta2, tb2)));
        return o;
    }
    // Two direction bytes of one word (low half, high half).
    __device__ __forceinline__ static uint32_t pack1(const DirWord &w)
    {
        const uint32_t b = __builtin_amdgcn_bitop3_b32(0x00070007u, w.z, w.f >> 8, RIGHT ? 0x3a : 0xca);
        return perm(b, b, 0x0c0c0200u);
    }
    // Four direction bytes of two words: (first.lo, second.lo, first.hi,
    // second.hi).
    __device__ __forceinline__ static uint32_t pack(const DirWord &first, const DirWord &second)
    {
        const uint32_t f = perm(second.f, first.f, 0x07030501u);
        const uint32_t z = perm(second.z, first.z, 0x06020400u);
        // right alignment: the index is the complement of the tag
        return __builtin_amdgcn_bitop3_b32(0x07070707u, z, f, RIGHT ? 0x3a : 0xca);
    }
};

struct RawCell {
    static constexpr int kScale = 1;
    static constexpr int p = 0;
    uint32_t e1, e2, l1, l2;
    int sm, sx;

    __device__ __forceinline__ RawCell(const KswScore &sc, bool)
    {
        e1 = splat(sc.e), e2 = splat(sc.e2), l1 = splat(sc.G1), l2 = splat(sc.G2);
        sm = -sc.mch, sx = -sc.mis;
    }
    __device__ __forceinline__ uint32_t x0() const { return l1; }
    __device__ __forceinline__ uint32_t x20() const { return l2; }
    __device__ __forceinline__ uint32_t y0() const { return l1; }
    __device__ __forceinline__ uint32_t y20() const { return l2; }
    __device__ __forceinline__ int diff(int w) const { return -w; }

    __device__ __forceinline__ DirWord step(uint32_t s, Down &d, Right &r) const
    {
        const uint32_t a = add2(d.x, d.v), b = add2(r.y, r.u), a2 = add2(d.x2, d.v), b2 = add2(r.y2, r.u);
        const uint32_t z = min3(min3(s, a, b), a2, b2);
        const uint32_t m1 = sub2(e1, z), m2 = sub2(e2, z);
        const uint32_t un = sub2(z, d.v);
        d.v = sub2(z, r.u), r.u = un;
        d.x = min2(add2(a, m1), l1), r.y = min2(add2(b, m1), l1);
        d.x2 = min2(add2(a2, m2), l2), r.y2 = min2(add2(b2, m2), l2);
        DirWord o;
        o.z = 0, o.f = 0;
        return o;
    }
    __device__ __forceinline__ static uint32_t pack(const DirWord &, const DirWord &) { return 0; }
};

}  // namespace cell

// What a pass stores per cell.
enum Mode { kDirs = 0, kScoreOnly = 1, kTracks = 2 };

// The cell of a mode and how far its sums are scaled (as a shift).
template <bool RIGHT, int MODE> struct CellOf {
    typedef cell::RawCell type;
    static constexpr int shift = 0;
};
template <bool RIGHT> struct CellOf<RIGHT, kDirs> {
    typedef cell::DirCell<RIGHT> type;
    static constexpr int shift = 3;
};
}  // namespace kswhip
