// fp32 values on the bf16 matrix cores of gfx950: the exact split of a value
// into three bf16 numbers, shared by the GEMM, convolution and attention
// kernels.
//
// x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid:
// three times 8 significant bits (plus the residuals' signs) hold the 24 bits
// of an fp32 number, and both subtractions are exact.  Of the nine products
// of two split values, lo.lo, lo.mid and mid.lo lie below 2^-25 of the whole
// and are left out; the other six are accumulated in fp32.  Against 64 bits
// on MI355X (normal values, relative 2-norm error of the sums of K products):
// K 64 1.1e-7, 512 1.2e-7 to 3.4e-7, 8192 2.5e-7 to 1.4e-6 (sums flushed
// every 32 to 64 of K, or one chain), the fp32 matrix cores 1.4e-7, 4.1e-7
// and 1.6e-6.  The bf16 ones run 16 times the fp32 rate (2060 against 154
// TFLOP/s from registers), so six products cost 0.45 of one fp32 product.
#ifndef ZN_SPLIT_H
#define ZN_SPLIT_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "zn_mfma_stage.h"

namespace {

typedef __bf16 zn_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 zn_bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t zn_u32x4 __attribute__((ext_vector_type(4)));
typedef float zn_f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Operands are multiplied by 2^24 before the split and sums by 2^-48 after
// it: the last bit of the smallest fp32 number is then 2^-125, so no part of
// any split is subnormal (the matrix cores would flush it).
constexpr float kSplitScale = 16777216.0f;
constexpr float kSplitUnscale = 1.0f / (16777216.0f * 16777216.0f);

// Two fp32 values to the three bf16 parts of each, packed (low half: x0).
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const float t0 = x0 * kSplitScale, t1 = x1 * kSplitScale;
    const zn_bf16x2 h = __builtin_convertvector((f2{t0, t1}), zn_bf16x2);
    const uint32_t hb = __builtin_bit_cast(uint32_t, h);
    const float r0 = t0 - __builtin_bit_cast(float, hb << 16), r1 = t1 - __builtin_bit_cast(float, hb & 0xffff0000u);
    const zn_bf16x2 m = __builtin_convertvector((f2{r0, r1}), zn_bf16x2);
    const uint32_t mb = __builtin_bit_cast(uint32_t, m);
    const float q0 = r0 - __builtin_bit_cast(float, mb << 16), q1 = r1 - __builtin_bit_cast(float, mb & 0xffff0000u);
    const zn_bf16x2 l = __builtin_convertvector((f2{q0, q1}), zn_bf16x2);
    hi = __builtin_bit_cast(uint32_t, h);
    mid = __builtin_bit_cast(uint32_t, m);
    lo = __builtin_bit_cast(uint32_t, l);
}

// Eight values to the fragments of their three parts.
__device__ __forceinline__ void split8(const float (&x)[8], zn_u32x4 (&w)[3]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t hi, mid, lo;
        split_pair(x[2 * e], x[2 * e + 1], hi, mid, lo);
        w[0][e] = hi;
        w[1][e] = mid;
        w[2][e] = lo;
    }
}

}  // namespace

#endif
