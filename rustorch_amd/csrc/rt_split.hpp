// f32 operands as three bf16 terms each, for products on the bf16 matrix cores at f32 accuracy.
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each rounded to nearest: the differences are
// exact, and 3 x 8 bits of significand hold all 24 of x (below 2^-109 the last term meets the smallest bf16: an
// absolute error of 2^-134; a workgroup that reads values so small goes by split_too_small or kSplitLeast).  A product
// x * y is then the six terms hh, hm, mh, hl, mm, lh; what is left out, ml + lm + ll, is below 2^-26 |x y|, less than
// half of an f32 rounding.  Every term is exact in the f32 accumulator of
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

// Four values on their way through the split, in five steps of two to six instructions: steps 0, 2 and 4 give the packed h, m
// and l of either pair.  No instruction needs the one ahead of it: a wave alone on its SIMD issues a vector instruction
// every 5 clocks where four chains alternate and every 8.6 in a single one (six of them behind a matrix instruction: 38 and
// 55 clocks).
struct SplitQuad {
    static constexpr int STEPS = 5;
    float r[4], u[4];
    __device__ __forceinline__ void step(int k, uint32_t& w0, uint32_t& w1) {
        if (k % 2 == 0) {
            w0 = __builtin_bit_cast(uint32_t, __builtin_convertvector((split_f32x2_t{r[0], r[1]}), split_bf16x2_t));
            w1 = __builtin_bit_cast(uint32_t, __builtin_convertvector((split_f32x2_t{r[2], r[3]}), split_bf16x2_t));
            if (k == 4) return;
            u[0] = bf16_lo(w0);
            u[2] = bf16_lo(w1);
            u[1] = bf16_hi(w0);
            u[3] = bf16_hi(w1);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] -= u[i];
        }
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

// One of the three planes of a tile of 32 rows in LDS, rows of 32 DT bf16 without padding.  The same plane serves as rows
// (16-byte reads of 16 rows at one slot) and, through the transposing reads, as columns (8 bytes of four rows, 64 bytes of
// a row side by side): the XOR of the 16-byte slot index spreads the sixteen rows over all banks and keeps the 64 bytes of
// four rows in four different quarters of them.
template <int DT>
struct SplitPlane {
    static constexpr int DPAD = 32 * DT, SIZE = 32 * DPAD;  // in elements
    static __device__ __forceinline__ int swizzle(int r) {
        return DT == 4 ? 4 * (r & 3) + ((r >> 2) & 3) : (DT == 2 ? 4 * ((r >> 1) & 1) + ((r >> 2) & 3) : ((r >> 2) & 3));
    }
    static __device__ __forceinline__ int at(int row, int slot) { return row * DPAD + 8 * (slot ^ swizzle(row)); }
    // A operand over the head dim: elements 16j + 8hh .. of row `col`
    static __device__ __forceinline__ bf16x8_t row_frag(const __bf16* plane, int j, int col, int hh) {
        return *(const bf16x8_t*)(plane + at(col, 2 * j + hh));
    }
    // A operand over the rows: column 32t + lane % 32, slot e of a lane row 16j + 4hh + 8 (e / 4) + e % 4 -- the order in which
    // the score-shaped accumulators hold their rows
    static __device__ __forceinline__ bf16x8_t col_frag(const __bf16* plane, int t, int j, int lane) {
        typedef short s16x4_t __attribute__((ext_vector_type(4)));
        const int l = lane & 15, row = (l >> 2) + 4 * (lane >> 5), slot = 4 * t + 2 * ((lane >> 4) & 1) + ((l & 3) >> 1);
        auto read = [&](int r) __attribute__((always_inline)) {
            const __bf16* const p = plane + at(r, slot) + 4 * (l & 1);
            return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(p)));
        };
        const u32x2_t lo = read(16 * j + row), hi = read(16 * j + 8 + row);
        return __builtin_bit_cast(bf16x8_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
    }
};

// A fixed place in the instruction order: what is written before it stays before it.
#define RT_ORDER() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ f32x16_t mfma_h(bf16x8_t a, bf16x8_t b, f32x16_t acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}

constexpr float kSplitMost = 0x1p30f;  // the magnitude from which on the split products are not used
// The same for values so small that the last term of the split would count (largest of a group of eight; zeros are fine).
__device__ __forceinline__ bool split_too_small(float group_max) { return group_max < 0x1p-80f && group_max > 0.0f; }
// ... and for single values of V: 2 (bits of |x|) - 1 of 2^-100, from which on the last term of x is no subnormal.  Where one
// is smaller the results decide: a value, and each of its products, loses 2^-126 at most, so that a result (before it is
// divided by the row sum) of 2^-80 of that sum is off by less than 2^-26 of itself at 2^16 keys.  A subnormal in V leaves
// every row on the split products whose results are not small themselves; turned away by the value alone it cost each
// workgroup that read it the f32 pass.  us, one in every head, before -> now, clean: causal B=1 H=8 N=2048 D=64 83.7 -> 44.2,
// 44.7; B=4 H=16 N=1024 D=64 239.9 -> 101.3, 101.0; causal D=128 272 -> 125, 126.  In a column of zeros, whose results it is,
// it costs the f32 pass behind the other (154 -> 240).
constexpr uint32_t kSplitLeast = ((uint32_t)(127 - 100) << 24) - 1u;
constexpr float kSplitLeastResult = 0x1p-80f;
// The larger magnitude; a NaN is not seen.
__device__ __forceinline__ float split_max(float m, float x) { return __builtin_fmaxf(m, __builtin_fabsf(x)); }

// A tile of 32 rows in f32 on its way through the 256 threads of a workgroup into LDS, zeros beyond D and the last row (kRepeat:
// copies of the last row, for query rows that meet a key that may be infinite): for the rows that are done once more.  16-byte loads; a row's start is 4 banks behind the one before it.
template <int DT>
struct F32Tile {
    static constexpr int CH = 8 * DT, LD = 32 * DT + 4, SIZE = 32 * LD;
    f32x4_t r[DT];
    template <bool kRepeat = false>
    __device__ __forceinline__ void load(const float* __restrict__ src, size_t pitch, int row0, int N, int D, int tid) {
#pragma unroll
        for (int n = 0; n < DT; n++) {
            const int idx = 256 * n + tid, row = kRepeat ? min(row0 + idx / CH, N - 1) : row0 + idx / CH, d = 4 * (idx % CH);
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
