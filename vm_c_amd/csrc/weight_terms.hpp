// weight_terms.hpp -- softmax weights as sums of 16-bit terms, one MFMA each, so
// that P V keeps the weights' fp32 precision whatever V's 16-bit type is.
//
// Three terms hold the 24 bits of an fp32 weight: bf16 has 8 bits a term at any
// exponent a weight takes; fp16 has 11, but nothing below 2^-24, so a weight is
// off by at most 2^-25 (the kernels scale weights by 2^15, or by 2^7 where the
// reference max may lag by 2^8: at most 2^-40 or 2^-32 of a weight of 1, where
// a row's sum is at least 1 and fp32 keeps 2^-24 of it).
#pragma once

#include "vmc_common.hpp"

namespace vmc {
namespace {

template <bool BF>
struct WeightTerms {
    static constexpr int n = 3;
    // term u of (a, b) packed in t[u]; a and b become what the terms leave out
    static __device__ __forceinline__ void split(float& a, float& b, uint32_t (&t)[n]) {
#pragma unroll
        for (int u = 0; u < n; ++u) {
            t[u] = (uint32_t)f32_to_half<BF>(a) | ((uint32_t)f32_to_half<BF>(b) << 16);
            a -= half_to_f32<BF>((uint16_t)(t[u] & 0xffffu));
            b -= half_to_f32<BF>((uint16_t)(t[u] >> 16));
        }
    }
};

}  // namespace
}  // namespace vmc
