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
    // acc += the 24-bit entries of four codes; planes: 3 x kP dwords, low bytes first
    static __device__ __forceinline__ void add_fixed24(uint32_t s, const uint32_t* planes, uint32_t& acc) {
        const uint32_t s7 = low3(s), m8 = bit3(s);
        const uint32_t b0 = look(planes, s, s7, m8), b1 = look(planes + kP, s, s7, m8),
                       b2 = look(planes + 2 * kP, s, s7, m8);
        acc = __builtin_amdgcn_udot4(b0, 0x01010101u, acc, false);
        acc += __builtin_amdgcn_udot4(b1, 0x01010101u, 0u, false) << 8;
        acc += __builtin_amdgcn_udot4(b2, 0x01010101u, 0u, false) << 16;
    }
};

}  // namespace

// c[i]^2 of the 2^bits centroids in 24-bit fixed point, as byte planes
// (3 x 2^bits / 4 dwords).  Returns the unit: the largest square is 2^24 - 1
// units, so a sum of 128 stays below 2^31.  Each entry is off by half a unit
// at most and the sum by 6 units or so (64 at most), 2^-22 (2^-18) of the
// largest square, where the sum is about 27 (3-bit) or 17 (4-bit) of them:
// the rounding of a 128-term fp32 sum.
inline float tq_fixed24_planes(const float* cent, int bits, uint32_t* planes) {
    const int n = 1 << bits, np = n / 4;
    double mx = 0.0;
    for (int i = 0; i < n; ++i) mx = fmax(mx, (double)cent[i] * cent[i]);
    const float unit = (float)(mx / 16777215.0 * (1.0 + 1e-7));
    for (int i = 0; i < 3 * np; ++i) planes[i] = 0;
    for (int i = 0; i < n; ++i) {
        uint32_t q = (uint32_t)(int64_t)rint((double)cent[i] * cent[i] / (double)unit);
        if (q > 0xffffffu) q = 0xffffffu;
        for (int b = 0; b < 3; ++b) planes[b * np + i / 4] |= ((q >> (8 * b)) & 255u) << (8 * (i & 3));
    }
    return unit;
}

}  // namespace vmc
