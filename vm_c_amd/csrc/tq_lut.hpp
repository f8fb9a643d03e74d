// tq_lut.hpp -- TurboQuant codes to fp16 by byte permutes.
//
// A block of codes takes at most 2^BITS distinct fp16 values.  Their low and
// high bytes are kept as byte planes (one v_perm_b32 picks four of eight
// bytes), so four codes cost four permutes (3-bit), or eight and two bit
// selects (4-bit), wherever their 16-bit values come from; an LDS gather pays
// an address and a conversion per code and waits for its bank conflicts.
#pragma once

#include <math.h>

#include "vmc_common.hpp"

namespace vmc {
namespace {

// 32 codes of BITS bits, little endian, as four words of 8 codes (3-bit: 24
// bits, the bits above are the next chunk's).
template <int BITS>
__device__ __forceinline__ void tq_chunks(const uint32_t* c, uint32_t (&x)[4]) {
    if constexpr (BITS == 3) {
        x[0] = c[0];
        x[1] = __builtin_amdgcn_alignbit(c[1], c[0], 24);
        x[2] = __builtin_amdgcn_alignbit(c[2], c[1], 16);
        x[3] = c[2] >> 8;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = c[i];
    }
}

// 8 codes -> one byte each: s[0] codes 0 .. 3, s[1] codes 4 .. 7.
template <int BITS>
__device__ __forceinline__ void tq_spread(uint32_t x, uint32_t (&s)[2]) {
    if constexpr (BITS == 3) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t y = (x >> (12 * u)) & 0xfffu;
            const uint32_t t = (y | (y << 10)) & 0x003f003fu;
            s[u] = (t | (t << 5)) & 0x07070707u;
        }
    } else {
        const uint32_t ev = x & 0x0f0f0f0fu, od = (x >> 4) & 0x0f0f0f0fu;
        s[0] = __builtin_amdgcn_perm(od, ev, 0x05010400u);
        s[1] = __builtin_amdgcn_perm(od, ev, 0x07030602u);
    }
}

template <int BITS>
struct TqLut {
    static constexpr int kN = 1 << BITS, kP = kN / 4;  // values, dwords of one byte plane
    uint32_t lo[kP], hi[kP];

    // bytes t[s.b] of a plane for the four bytes s.b < kN of s
    static __device__ __forceinline__ uint32_t look(const uint32_t* t, uint32_t s, uint32_t s7, uint32_t m8) {
        if constexpr (BITS == 3) {
            return __builtin_amdgcn_perm(t[1], t[0], s);
        } else {
            const uint32_t a = __builtin_amdgcn_perm(t[1], t[0], s7), b = __builtin_amdgcn_perm(t[3], t[2], s7);
            return (m8 & b) | (~m8 & a);
        }
    }
    // 4-bit codes: the low three bits, and 0xff in the bytes with bit 3 set
    static __device__ __forceinline__ uint32_t low3(uint32_t s) { return BITS == 3 ? s : s & 0x07070707u; }
    static __device__ __forceinline__ uint32_t bit3(uint32_t s) {
        if constexpr (BITS == 3) return 0;
        const uint32_t b = (s >> 3) & 0x01010101u;
        return (b << 8) - b;
    }

    // the values fp16(base[i] * f + add), in byte planes
    __device__ __forceinline__ void build(const float* base, float f, float add) {
#pragma unroll
        for (int i = 0; i < kP; ++i) {
            uint32_t w[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
                w[u] = (uint32_t)f32_to_f16_bits(__builtin_fmaf(base[4 * i + 2 * u], f, add)) |
                       ((uint32_t)f32_to_f16_bits(__builtin_fmaf(base[4 * i + 2 * u + 1], f, add)) << 16);
            lo[i] = __builtin_amdgcn_perm(w[1], w[0], 0x06040200u);
            hi[i] = __builtin_amdgcn_perm(w[1], w[0], 0x07050301u);
        }
    }
    // the fp16 values of four codes (one a byte), two per dword
    __device__ __forceinline__ u32x2 pick(uint32_t s) const {
        const uint32_t s7 = low3(s), m8 = bit3(s);
        const uint32_t l = look(lo, s, s7, m8), h = look(hi, s, s7, m8);
        return u32x2{__builtin_amdgcn_perm(h, l, 0x05010400u), __builtin_amdgcn_perm(h, l, 0x07030602u)};
    }
    // acc[b] += byte b of the 32-bit entries of four codes; planes: 4 x kP
    // dwords, low bytes first
    static __device__ __forceinline__ void add_squares(uint32_t s, const uint32_t* planes, uint32_t (&acc)[4]) {
        const uint32_t s7 = low3(s), m8 = bit3(s);
#pragma unroll
        for (int b = 0; b < 4; ++b)
            acc[b] = __builtin_amdgcn_udot4(look(planes + b * kP, s, s7, m8), 0x01010101u, acc[b], false);
    }
};

// The sum of a K row's 128 entries in units, for lanes 0 .. 31 and 32 on alike:
// sel holds 32 codes of it in each of four lanes below 32 (a quad), one a byte.
// The lane 32 on takes half of them (its own are V's): 2048 tokens over a
// 30720-token prefix of 4-bit slots 1547 us, 1689 with every lane looking up all
// 32.  Integers keep the sum exact (each half word's below 2^23) up to the one
// rounding here.
template <int BITS>
__device__ __forceinline__ float tq_row_squares(const uint32_t (&sel)[4][2], const uint32_t* planes, int lane) {
    uint32_t acc[4] = {};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t mine = sel[j][0], theirs = sel[j][1];
        swap_pair32(mine, theirs);  // lanes 32 on: sel[j][1] of 32 lanes below
        TqLut<BITS>::add_squares(mine, planes, acc);
    }
    uint32_t w[2] = {(acc[1] << 8) + acc[0], (acc[3] << 8) + acc[2]};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        w[i] += row_xor_u32<1>(w[i], lane);
        w[i] += row_xor_u32<2>(w[i], lane);
        uint32_t o = w[i];
        swap_pair32(w[i], o);
        w[i] += o;
    }
    return __builtin_fmaf((float)w[1], 65536.0f, (float)w[0]);
}

}  // namespace

// c[i]^2 of the 2^bits centroids in 32-bit fixed point, as byte planes
// (2^bits entries: 2^bits dwords).  Returns the unit: the largest square is
// 2^32 - 1 of them.  An entry is off by half a unit at most, 2^-24 of the
// smallest square (4-bit; 3-bit 2^-28): no more than a squared fp32 centroid's
// own rounding, and the sum itself is exact where fp32 rounds at each term.
inline float tq_square_planes(const float* cent, int bits, uint32_t* planes) {
    const int n = 1 << bits, np = n / 4;
    double mx = 0.0;
    for (int i = 0; i < n; ++i) mx = fmax(mx, (double)cent[i] * cent[i]);
    const float unit = (float)(mx / 4294967295.0 * (1.0 + 1e-7));
    for (int i = 0; i < 4 * np; ++i) planes[i] = 0;
    for (int i = 0; i < n; ++i) {
        double q = rint((double)cent[i] * cent[i] / (double)unit);
        if (q > 4294967295.0) q = 4294967295.0;
        for (int b = 0; b < 4; ++b) planes[b * np + i / 4] |= (((uint32_t)q >> (8 * b)) & 255u) << (8 * (i & 3));
    }
    return unit;
}

}  // namespace vmc
