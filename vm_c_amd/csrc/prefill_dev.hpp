// prefill_dev.hpp -- device pieces the prefill kernels share: the 32x32 MFMA of
// one 16-bit type and the load-to-LDS transfers.
#pragma once

#include "vmc_common.hpp"

namespace vmc {
namespace {

template <bool BF16>
struct MT;
template <>
struct MT<true> {
    using v8 = bf16x8;
    static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint16_t cvt(float x) { return f32_to_bf16_bits(x); }
};
template <>
struct MT<false> {
    using v8 = f16x8;
    static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint16_t cvt(float x) { return f32_to_f16_bits(x); }
};

template <typename V8>
__device__ __forceinline__ V8 as_v8(u32x4 w) {
    return __builtin_bit_cast(V8, w);
}

// One 16-byte-per-lane load-to-LDS transfer: lane L's 16 bytes from src land
// at LDS address m0 + 16 L.  Issued from asm so the compiler does not track it: it
// would otherwise make every later LDS read wait for all transfers in
// flight (it cannot tell the slots apart); the kernel waits for them itself.
__device__ __forceinline__ void dma16m(const void* src, uint32_t m0) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "{m0}"(m0) : "memory");
}
// The same transfer from a wave-uniform base (SGPRs) plus a 32-bit per-lane
// offset: no per-lane 64-bit address arithmetic.
__device__ __forceinline__ void dma16s(const void* base, uint32_t off, uint32_t m0) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(m0) : "memory");
}

}  // namespace
}  // namespace vmc
