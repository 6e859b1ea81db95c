// The two-term f16 split x = hi + lo (hi = f16(x), lo = f16(x - hi)) that feeds the 16-bit matrix
// units with f32 operands: 22 of x's 24 significand bits.  Four VALU instructions per pair: one
// v_cvt_pk_f16_f32 rounds the pair; v_fma_mix_f32 reads each half as f16 and forms x - hi in f32 in
// one instruction (exact: hi is x rounded, so x - hi is representable); a second v_cvt_pk rounds
// the remainders.  (The compiler's own lowering of the same expressions converts every element
// twice: 8 per pair.)
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace zwg_split {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sub_f16_lo(uint32_t pair, float x) { // x - (float)low half of pair
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(x));
    return r;
}
__device__ __forceinline__ float sub_f16_hi(uint32_t pair, float x) { // x - (float)high half of pair
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(x));
    return r;
}
__device__ __forceinline__ uint32_t split2_f16(float a, float b, uint32_t &lo) {
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){sub_f16_lo(h, a), sub_f16_hi(h, b)}, f16x2));
    return h;
}
__device__ __forceinline__ void split8(const f32x8 &x, f16x8 &hi, f16x8 &lo) {
    u32x4 h, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t li;
        h[i] = split2_f16(x[2 * i], x[2 * i + 1], li);
        l[i] = li;
    }
    hi = __builtin_bit_cast(f16x8, h);
    lo = __builtin_bit_cast(f16x8, l);
}
__device__ __forceinline__ void split4(const f32x4 &x, f16x4 &hi, f16x4 &lo) {
    u32x2 h, l;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t li;
        h[i] = split2_f16(x[2 * i], x[2 * i + 1], li);
        l[i] = li;
    }
    hi = __builtin_bit_cast(f16x4, h);
    lo = __builtin_bit_cast(f16x4, l);
}

} // namespace zwg_split
