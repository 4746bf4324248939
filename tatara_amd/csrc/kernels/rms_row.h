// The arithmetic of the RMS row norm (rms_only.metal:5-43), shared by the norm kernel and
// by the projections that apply the norm while they stage their input rows, so that both
// produce the same bits: four squares summed in order per 4-value slice, slices summed by
// the adjacent-pairs tree, out = bf16(w * bf16(x * inverse)).
#pragma once

#include <stdint.h>

#include <hip/hip_runtime.h>

#include "../tt_constants.h"

namespace tt {

__device__ __forceinline__ float rms_widen(uint16_t h) {
    return __uint_as_float(static_cast<uint32_t>(h) << 16);
}
// round to nearest even with subnormal results flushed to signed zero
__device__ __forceinline__ uint16_t rms_store16(float v) {
    uint32_t b = __float_as_uint(v);
    if ((b & 0x7F800000u) == 0) b &= 0x80000000u;
    if ((b & 0x7F800000u) == 0x7F800000u) return static_cast<uint16_t>(b >> 16);
    const uint16_t h = static_cast<uint16_t>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
    return (h & 0x7F80u) ? h : static_cast<uint16_t>(h & 0x8000u);
}
__device__ __forceinline__ uint16_t rms_fz16(uint16_t h) {
    return (h & 0x7F80u) ? h : static_cast<uint16_t>(h & 0x8000u);
}

// squares of a slice of four values (two packed dwords), summed in order
__device__ __forceinline__ float rms_slice_squares(uint32_t low, uint32_t high) {
    const float x0 = __uint_as_float(low << 16), x1 = __uint_as_float(low & 0xFFFF0000u);
    const float x2 = __uint_as_float(high << 16), x3 = __uint_as_float(high & 0xFFFF0000u);
    float sum = 0.0f;
    sum += x0 * x0;
    sum += x1 * x1;
    sum += x2 * x2;
    sum += x3 * x3;
    return sum;
}

__device__ __forceinline__ float rms_inverse(float total, uint32_t hidden) {
    return 1.0f / sqrtf(total / static_cast<float>(hidden) + kRmsNormEpsilon);
}

// a magnitude below the normal range to signed zero
__device__ __forceinline__ float rms_flush(float v) {
    return fabsf(v) < 0x1p-126f ? __uint_as_float(__float_as_uint(v) & 0x80000000u) : v;
}
// rms_store16 of two values, packed, by the hardware's conversion (round to nearest even; a value
// that is not subnormal does not round to one; the NaN of a sum or a product is quiet already and keeps
// its upper bits)
__device__ __forceinline__ uint32_t rms_store_pair(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float Pair;
    typedef __attribute__((ext_vector_type(2))) __bf16 Rounded;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(Pair{rms_flush(a), rms_flush(b)}, Rounded));
}
__device__ __forceinline__ float rms_low(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float rms_high(uint32_t pair) { return __uint_as_float(pair & 0xFFFF0000u); }

// two values of a row and their weights, packed: bf16(w * bf16(x * inverse)) of each
__device__ __forceinline__ uint32_t rms_scale_pair(uint32_t x_pair, uint32_t w_pair, float inverse) {
    const uint32_t scaled = rms_store_pair(rms_low(x_pair) * inverse, rms_high(x_pair) * inverse);
    return rms_store_pair(rms_flush(rms_low(w_pair)) * rms_low(scaled),
                          rms_flush(rms_high(w_pair)) * rms_high(scaled));
}
// the residual sum of two pairs: bf16(a + b) of each
__device__ __forceinline__ uint32_t rms_add_pair(uint32_t a_pair, uint32_t b_pair) {
    return rms_store_pair(rms_flush(rms_low(a_pair)) + rms_flush(rms_low(b_pair)),
                          rms_flush(rms_high(a_pair)) + rms_flush(rms_high(b_pair)));
}

}  // namespace tt
