// f32 operands as three bf16 terms each, for products on the bf16 matrix cores at f32 accuracy.
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each rounded to nearest: the differences are
// exact, and 3 x 8 bits of significand hold all 24 of x (below 2^-109 the last term meets the smallest bf16: an
// absolute error of 2^-134; a workgroup that reads a group of values below 2^-80 goes by split_too_small).  A product x * y is then the six terms hh, hm, mh, hl, mm, lh; what is left out, ml + lm + ll,
// is below 2^-26 |x y|, less than half of an f32 rounding.  Every term is exact in the f32 accumulator of
// v_mfma_f32_32x32x16_bf16, whose rate is 16 times that of v_mfma_f32_32x32x2_f32: six of them are 2.7 times the f32 rate.
//
// NaN survives the split as three NaN, and whatever f32 arithmetic makes NaN of it comes out NaN here.  Infinities do not
// (inf - inf), and finite values whose products overflow f32 would give inf - inf where one product gives inf.  The
// kernels keep the largest magnitude of everything they split: below 2^30 neither can happen, in a product of two nor in
// the gradients' products of three.  A workgroup that finds one above it does its rows once more on the f32 matrix cores.
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

constexpr float kSplitMost = 0x1p30f;  // the magnitude from which on the split products are not used
// The same for values so small that the last term of the split would count (largest of a group of eight; zeros are fine).
__device__ __forceinline__ bool split_too_small(float group_max) { return group_max < 0x1p-80f && group_max > 0.0f; }
// The larger magnitude; a NaN is not seen.
__device__ __forceinline__ float split_max(float m, float x) { return __builtin_fmaxf(m, __builtin_fabsf(x)); }

// A tile of 32 rows in f32 on its way through the 256 threads of a workgroup into LDS, zeros beyond the last row and D: for
// the rows that are done once more.  16-byte loads; a row's start is 4 banks behind the one before it.
template <int DT>
struct F32Tile {
    static constexpr int CH = 8 * DT, LD = 32 * DT + 4, SIZE = 32 * LD;
    f32x4_t r[DT];
    __device__ __forceinline__ void load(const float* __restrict__ src, size_t pitch, int row0, int N, int D, int tid) {
#pragma unroll
        for (int n = 0; n < DT; n++) {
            const int idx = 256 * n + tid, row = row0 + idx / CH, d = 4 * (idx % CH);
            f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
            if (row < N && d < D) z = *(const f32x4_t*)(src + (size_t)row * pitch + d);
            r[n] = z;
        }
    }
    __device__ __forceinline__ void store(float* dst, int tid) const {
#pragma unroll
        for (int n = 0; n < DT; n++) {
            const int idx = 256 * n + tid;
            *(f32x4_t*)(dst + (idx / CH) * LD + 4 * (idx % CH)) = r[n];
        }
    }
};

// acc += X . Y^T over the head dim, in the order of the f32 kernels (d = 8j + 4 hh + i): row `col` of a tile in LDS as A
// operand, y[4j + i] in registers as B.
template <int DT>
__device__ __forceinline__ void f32_rows(f32x16_t& acc, const float* tile, const float (&y)[16 * DT], int col, int hh) {
#pragma unroll
    for (int j = 0; j < 4 * DT; j++) {
        const f32x4_t a = *(const f32x4_t*)(tile + col * F32Tile<DT>::LD + 8 * j + 4 * hh);
#pragma unroll
        for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], y[4 * j + i], acc, 0, 0, 0);
    }
}
// acc[t] += X^T . w over the tile's rows: column 32t + col of the tile, w as a score accumulator holds it
template <int DT>
__device__ __forceinline__ void f32_cols(f32x16_t (&acc)[DT], const float* tile, const f32x16_t& w, int col, int hh) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float* row = tile + (8 * (i >> 2) + 4 * hh + (i & 3)) * F32Tile<DT>::LD + col;
#pragma unroll
        for (int t = 0; t < DT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(row[32 * t], w[i], acc[t], 0, 0, 0);
    }
}
// The B operand of f32_rows: this lane's elements of a row, zeros beyond D and where `ok` is false.
template <int DT>
__device__ __forceinline__ void f32_row(float (&y)[16 * DT], const float* __restrict__ row, bool ok, int D, int hh) {
#pragma unroll
    for (int j = 0; j < 4 * DT; j++) {
        f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
        if (ok && 8 * j + 4 * hh < D) z = *(const f32x4_t*)(row + 8 * j + 4 * hh);
#pragma unroll
        for (int i = 0; i < 4; i++) y[4 * j + i] = z[i];
    }
}

}  // namespace rt
