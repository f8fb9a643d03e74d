// generic_row.hpp -- the one-wave attention row: online softmax and O += p V in
// fp32 over any K/V source, one key per lane.  gen_attn_kernel is this loop
// over a whole row; the MFMA kernels of head_dim 64 and 256 rerun a row with
// it when their products met an infinity or a NaN (an MFMA multiplies every
// key's V by its weight, also where the weight is 0).
#pragma once

#include "generic_attn.hpp"
#include "vmc_common.hpp"
#include "vmc_tq.hpp"

namespace vmc {
namespace {

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, shfl_xor(v, m));
    return v;
}
__device__ __forceinline__ float wave_min_f(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fminf(v, shfl_xor(v, m));
    return v;
}
__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += shfl_xor(v, m);
    return v;
}

// fp8 key byte -> float (fp8_e4m3_to_float / fp8_e4b15_to_float,
// turboquant_kernels.cu:85-96, :136-143): (1 + m/8) 2^(e - bias), zero codes
// signed zero
__device__ __forceinline__ float fp8_decode(uint32_t b, int e4b15) {
    const uint32_t e = (b >> 3) & 0xfu, m = b & 7u;
    float v = 0.0f;
    if (e != 0 || m != 0) v = ldexpf(1.0f + (float)m * 0.125f, (int)e - (e4b15 ? 15 : 7));
    return (b & 0x80u) ? -v : v;
}

// codes 8g .. 8g+7 of a packed TurboQuant code array (2-byte aligned):
// 4-bit -> 4 bytes at 4g (even d low nibble), 3-bit -> 3 bytes at 3g, code
// i at bits 3i; returned as a word with code i at bits BITS * i
template <int BITS>
__device__ __forceinline__ uint32_t codes8(const uint8_t* p, int g) {
    if constexpr (BITS == 4) {
        return ld_u16(p + 4 * g) | (ld_u16(p + 4 * g + 2) << 16);
    } else {
        const int o = 3 * g, a = o & ~1;
        const uint32_t w = ld_u16(p + a) | (ld_u16(p + a + 2) << 16);
        return (w >> (8 * (o & 1))) & 0xffffffu;
    }
}
template <int BITS>
__device__ __forceinline__ uint32_t code_at(const uint8_t* p, int d) {
    if constexpr (BITS == 4) {
        return (p[d >> 1] >> (4 * (d & 1))) & 0xfu;
    } else {
        return (codes8<3>(p, d >> 3) >> (3 * (d & 7))) & 7u;
    }
}

template <bool BF>
__device__ __forceinline__ float ld_half(const uint8_t* p) {
    return half_to_f32<BF>((uint16_t)ld_u16(p));
}

// Keys k_begin .. n - 1 of one row against q (qs: fp32, in LDS; rotated for
// TurboQuant codebook keys).  key_at(k, ke, ve) sets key k's K and V entries
// and says whether it is there (false: a block-table hole).  Leaves the
// reference max m (natural log units), the sum l and this lane's output
// dims lane + 64 i, unnormalised.  One wave; results of m and l in every lane.
template <int D, int SRC, int KB, int VB, bool BF, typename KeyAt>
__device__ __forceinline__ void gen_row(const GenArgs& a, const TQTables& tab, const float* qs, int lane, int k_begin,
                                        int n, KeyAt key_at, float& m, float& l, float (&acc)[D / 64]) {
    constexpr int NPL = D / 64;
    m = -__builtin_inff();
    l = 0.0f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) acc[i] = 0.0f;
    for (int k0 = k_begin; k0 < n; k0 += 64) {
        const int kk = k0 + lane;
        const uint8_t* ke = nullptr;
        const uint8_t* ve = nullptr;
        bool valid = kk < n;
        if (valid) valid = key_at(kk, ke, ve);
        // ---- score of this lane's key
        float s = -__builtin_inff();
        if (valid) {
            float dot = 0.0f;
            if constexpr (SRC == GEN_F16 || SRC == GEN_BF16 || SRC == GEN_LOCAL) {
                constexpr bool KBF = SRC == GEN_BF16 || (SRC == GEN_LOCAL && BF);
                for (int d = 0; d < D; d += 2) {
                    const uint32_t wv = *reinterpret_cast<const uint32_t*>(ke + 2 * d);
                    dot = __builtin_fmaf(qs[d], half_to_f32<KBF>((uint16_t)(wv & 0xffffu)), dot);
                    dot = __builtin_fmaf(qs[d + 1], half_to_f32<KBF>((uint16_t)(wv >> 16)), dot);
                }
            } else if constexpr (SRC == GEN_Q8 || SRC == GEN_Q4) {
                constexpr int BE = SRC == GEN_Q8 ? 34 : 18;
                for (int b = 0; b < D / 32; ++b) {
                    const uint8_t* blk = ke + BE * b;
                    const float db = ld_half<false>(blk);
                    float part = 0.0f;
                    for (int j = 0; j < 32; ++j) {
                        int x;
                        if constexpr (SRC == GEN_Q8) x = (int)(int8_t)blk[2 + j];
                        else x = (int)((blk[2 + (j & 15)] >> (j < 16 ? 0 : 4)) & 0xf) - 8;
                        part = __builtin_fmaf(qs[32 * b + j], (float)x, part);
                    }
                    dot = __builtin_fmaf(db, part, dot);
                }
            } else if constexpr (KB == 8) {
                // fp8 keys: q not rotated, no norm
                for (int d = 0; d < D; ++d) dot = __builtin_fmaf(qs[d], fp8_decode(ke[d], a.fp8_e4b15), dot);
            } else {
                // codebook keys: C[code] / ||C[codes]|| * norm (tq_decode_stage1 :416-450)
                float cn = 0.0f;
                for (int gq = 0; gq < D / 8; ++gq) {
                    const uint32_t cw = codes8<KB>(ke, gq);
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float cv = tab.centroids[(cw >> (KB * i)) & ((1u << KB) - 1)];
                        dot = __builtin_fmaf(qs[8 * gq + i], cv, dot);
                        cn = __builtin_fmaf(cv, cv, cn);
                    }
                }
                const float ci = a.norm_correction ? 1.0f / sqrtf(cn + 1e-16f) : 1.0f;
                dot = dot * ci * ld_half<BF>(ke + a.mse_bytes);
            }
            s = dot * a.scale;
        }
        // ---- online softmax over the 64 keys
        const float mc = wave_max_f(s);
        const float m_new = fmaxf(m, mc);
        if (m_new == -__builtin_inff()) continue;  // no key so far (uniform)
        const float alpha = expf(m - m_new);  // 0 from -inf
        const float p = valid ? expf(s - m_new) : 0.0f;
        l = l * alpha + wave_sum_f(p);
#pragma unroll
        for (int i = 0; i < NPL; ++i) acc[i] *= alpha;
        m = m_new;
        // ---- O += p V: lane owns dims lane + 64 i
        const uintptr_t vaddr = (uintptr_t)ve;
        for (int j = 0; j < 64 && k0 + j < n; ++j) {
            const float pj = shfl(p, j);
            if (pj == 0.0f) continue;  // masked, a hole, or underflow (uniform)
            const uint32_t lo32 = (uint32_t)__shfl((int)(uint32_t)vaddr, j, kWave);
            const uint32_t hi32 = (uint32_t)__shfl((int)(uint32_t)(vaddr >> 32), j, kWave);
            const uint8_t* vj = reinterpret_cast<const uint8_t*>(((uint64_t)hi32 << 32) | lo32);
            float vs = 0.0f, vz = 0.0f;
            if constexpr (SRC == GEN_TQ) {
                vs = ld_half<BF>(vj + a.key_packed + a.val_data);
                vz = ld_half<BF>(vj + a.key_packed + a.val_data + 2);
            }
#pragma unroll
            for (int i = 0; i < NPL; ++i) {
                const int d = lane + 64 * i;
                float v;
                if constexpr (SRC == GEN_F16 || SRC == GEN_BF16 || SRC == GEN_LOCAL) {
                    constexpr bool VBF = SRC == GEN_BF16 || (SRC == GEN_LOCAL && BF);
                    v = ld_half<VBF>(vj + 2 * d);
                } else if constexpr (SRC == GEN_Q8) {
                    const uint8_t* blk = vj + 34 * (d >> 5);
                    v = ld_half<false>(blk) * (float)(int8_t)blk[2 + (d & 31)];
                } else if constexpr (SRC == GEN_Q4) {
                    const uint8_t* blk = vj + 18 * (d >> 5);
                    const int j5 = d & 31;
                    v = ld_half<false>(blk) * (float)((int)((blk[2 + (j5 & 15)] >> (j5 < 16 ? 0 : 4)) & 0xf) - 8);
                } else {
                    v = __builtin_fmaf((float)code_at<VB>(vj + a.key_packed, d), vs, vz);
                }
                acc[i] = __builtin_fmaf(pj, v, acc[i]);
            }
        }
    }
}

}  // namespace
}  // namespace vmc
