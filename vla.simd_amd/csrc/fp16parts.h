// fp16parts.h - a float as two fp16 parts, for fp32 products on the fp16 matrix
// cores.
//
// Scaled by a power of two, x = h + m + e with h = fp16(x), m = fp16(x - h) and
// |e| <= 2^-22 |x| or 2^-25 (half of fp16's smallest step), whichever is more.
// A product of two floats is hh + hm + mh to that accuracy. The scales keep the
// largest value below 2^15 (fp16 ends at 65504), so what shares one loses no
// more than 2^-40 of the largest.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vla {
namespace hip {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// The two parts of x0 and x1, packed. (v_fma_mix{lo,hi}_f16 would scale, round
// and subtract at once, but they issue at half rate: 8 cycles against 4 for
// v_cvt_pk_f16_f32 and v_fma_mix_f32.)
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& m) {
    float r0, r1;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(h) : "v"(x0), "v"(x1));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(h), "v"(x0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(h), "v"(x1));
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(m) : "v"(r0), "v"(r1));
}

// max(m, |x|, |y|); NaN is passed over
__device__ __forceinline__ float absmax(float m, float x, float y) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(x), "v"(y));
    return m;
}
__device__ __forceinline__ float absmax4(float m, const float4& v) { return absmax(absmax(m, v.x, v.y), v.z, v.w); }

// The power of two that brings `mx` to [2^top, 2^(top + 1)), as its biased
// exponent, kept where it and its inverse (254 minus it) are normal floats.
__device__ __forceinline__ uint32_t scale_exp(float mx, int top) {
    const int e = 254 + top - (int)((__float_as_uint(mx) >> 23) & 0xffu);
    return (uint32_t)(e < 1 ? 1 : e > 253 ? 253 : e);
}
__device__ __forceinline__ float exp_float(uint32_t e) { return __uint_as_float(e << 23); }

}  // namespace hip
}  // namespace vla
