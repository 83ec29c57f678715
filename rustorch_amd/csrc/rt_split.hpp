// f32 operands as three bf16 terms each, for products on the bf16 matrix cores at f32 accuracy.
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each rounded to nearest: the differences are
// exact, and 3 x 8 bits of significand hold all 24 of x (below 2^-109 the last term meets the smallest bf16: an
// absolute error of 2^-134; a workgroup that reads a group of values below 2^-80 goes by split_too_small).  A product x * y is then the six terms hh, hm, mh, hl, mm, lh; what is left out, ml + lm + ll,
// is below 2^-26 |x y|, less than half of an f32 rounding.  Every term is exact in the f32 accumulator of
// v_mfma_f32_32x32x16_bf16, whose rate is 16 times that of v_mfma_f32_32x32x2_f32: six of them are 2.7 times the f32 rate.
//
// Infinities and NaN do not survive the split (inf - inf), and finite values whose products overflow f32 would give
// inf - inf where one product gives inf.  The kernels sum the squares of everything they split: below 2^60 no
// operand exceeds 2^30 and neither can happen, in a product of two nor in the gradients' products of three.  A workgroup
// that finds the sum above it, or NaN, does its rows once more on the f32 matrix cores.
#pragma once
#include "rt_common.hpp"

namespace rt {

typedef __bf16 split_bf16x2_t __attribute__((ext_vector_type(2)));
typedef float split_f32x2_t __attribute__((ext_vector_type(2)));

struct Split8 {
    bf16x8_t p[3];  // h, m, l
};

// Two values on their way through the split: step n = 0, 1, 2 gives the packed h, m and l.  Five vector instructions a
// step fit between two matrix instructions of one wave.
struct SplitPair {
    split_f32x2_t r;
    __device__ __forceinline__ uint32_t step(int n) {
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, split_bf16x2_t));
        if (n < 2) {
            r[0] -= bf16_lo(w);
            r[1] -= bf16_hi(w);
        }
        return w;
    }
};

__device__ __forceinline__ void split2(float x0, float x1, uint32_t (&w)[3]) {
    SplitPair s{{x0, x1}};
#pragma unroll
    for (int n = 0; n < 3; n++) w[n] = s.step(n);
}

__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
    u32x4_t w[3];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        uint32_t u[3];
        split2(x[2 * e], x[2 * e + 1], u);
#pragma unroll
        for (int n = 0; n < 3; n++) w[n][e] = u[n];
    }
    Split8 s;
#pragma unroll
    for (int n = 0; n < 3; n++) s.p[n] = __builtin_bit_cast(bf16x8_t, w[n]);
    return s;
}

// A fixed place in the instruction order: what is written before it stays before it.
#define RT_ORDER() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ f32x16_t mfma_h(bf16x8_t a, bf16x8_t b, f32x16_t acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}

constexpr float kSplitMost = 0x1p60f;  // the sum of squares from which on the split products are not used
// The same for values so small that the last term of the split would count (largest of a group of eight; zeros are fine).
__device__ __forceinline__ bool split_too_small(float group_max) { return group_max < 0x1p-80f && group_max > 0.0f; }

}  // namespace rt
