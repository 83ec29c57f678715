// Gradients of f32 attention on the bf16 matrix cores, every operand as three bf16 terms (rt_split.hpp): the two kernels of
// flash_bwd_f32.hip (its header has the formulas) for launches with enough rows to fill the chip with 128 a workgroup.
//
// A wave owns 32 rows (keys for dK/dV, queries for dQ), split once into registers as B operands; the four waves of a
// workgroup walk the same tiles of 32 rows of the other side, which the workgroup splits once into LDS: planes of rows, read as
// rows (A operand of the score-shaped products) and, where a gradient contracts over them, as columns by the transposing reads
// (A operand of dV^T += dO^T P and the like, in the order the weights sit in the accumulators).  Every output row has one
// owner: no atomics, the same bits on every launch.
//
// What bounds them: a wave takes the register file of its SIMD (400 registers at head dim 64), so nothing covers what it waits
// for; at head dim 64 a tile is 96 (dK/dV) and 72 (dQ) matrix instructions of 32 clocks and 520 and 400 vector ones of 4, each
// kernel with room to run the one beside the other, and takes 4400 and 3500 clocks.  Hence: vector work between all matrix
// instructions, in runs of independent instructions (SplitQuad); LDS writes one at a time; nothing loaded is looked at in
// the step that requests it, nor copied there; owners pinned to the accumulation registers, where the matrix instructions read them
// and no vector instruction wants them; sums wherever the vector unit need not fetch them.  Time of both, B=4 H=16 N=1024 D=64: f32 kernels 506 us, this form with columns of its
// own in LDS 362, with the transposing reads 341, with every vector step beside a matrix instruction 336, without a wait
// for the row statistic where it is requested 327, sums pinned 321, dQ in the same order 312, independent runs and single
// writes 308.  B=2 N=2048 973, 689, 583; head dim 32 273, 214, 171.  (dQ with two waves a SIMD, 40 registers spilled: 318.)  On another
// card: tiles loaded without a branch and owners all at once 327 -> 318, sums not pinned 313; 2 x 12 heads N=400 39.3 -> 37.1.
// Relative error against 64 bits 5.9e-7 -> 4.5e-7, 7.3e-7 -> 5.9e-7, 5.5e-7 -> 4.4e-7 (f32 kernels -> this).
#include <type_traits>

#include "rt_common.hpp"
#include "rt_kernels.hpp"
#include "rt_split.hpp"

namespace rt {

namespace {

#define RT_INLINE __attribute__((always_inline))  // lambdas over the wave's registers: a call would put them in memory

constexpr int kTile = 32;
constexpr int kTermA[6] = {2, 1, 1, 0, 0, 0}, kTermB[6] = {0, 1, 0, 2, 1, 0};  // planes of the six terms, small ones first

__device__ __forceinline__ void zero16(f32x16_t& x) {
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = 0.0f;
}

// what the split does not carry raises the largest magnitude to kSplitMost (rt_split.hpp)
__device__ __forceinline__ void check8(const float (&x)[8], float& chk) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) m = split_max(m, x[i]);
    chk = split_too_small(m) ? kSplitMost : __builtin_fmaxf(chk, m);
}

// One streamed matrix [N, D]: a tile's rows on their way from memory into LDS, in pieces of eight elements of a row, kN a thread.
// Rows behind the last repeat it; whoever reads the tile gives them weights of zero.
template <int DT>
struct Stream {
    using Plane = SplitPlane<DT>;
    static constexpr int DPAD = 32 * DT, CH = DPAD / 8, ITEMS = kTile * CH, kN = (ITEMS + 255) / 256;
    static constexpr int SIZE = 3 * Plane::SIZE;  // bf16 elements of a tile
    f32x4_t r[kN][2];
    __amdgpu_buffer_rsrc_t rs;
    int pitch, last;

    // Where a thread's pieces lie in a row: byte offsets of either half, past every descriptor where the row has no such elements or the
    // tile no such piece.
    struct Place {
        uint32_t at[kN][2];
        __device__ __forceinline__ Place(int D, int tid) {
#pragma unroll
            for (int n = 0; n < kN; n++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int d = 8 * ((256 * n + tid) % CH) + 4 * u;
                    at[n][u] = has(n, tid) && d < D ? 4u * (uint32_t)d : 0x80000000u;
                }
        }
    };
    static __device__ __forceinline__ bool has(int n, int tid) { return ITEMS % 256 == 0 || 256 * n + tid < ITEMS; }

    // (N rows of D f32, less than 2 GiB)
    __device__ __forceinline__ Stream(const float* src, int N, int D)
        : rs(__builtin_amdgcn_make_buffer_rsrc((void*)src, 0, 4u * (uint32_t)N * (uint32_t)D, kBufferFlags)), pitch(4 * D), last(N - 1) {
#pragma unroll
        for (int n = 0; n < kN; n++) r[n][0] = r[n][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // Without a branch around a load, or two ways to one: where those met, the registers were copied, and the copies waited for the
    // loads just requested.
    __device__ __forceinline__ void load(int tile, const Place& place, int tid) {
        const int row0 = min(kTile * tile, last), left = last - row0;
        const uint32_t so = (uint32_t)row0 * (uint32_t)pitch;
#pragma unroll
        for (int n = 0; n < kN; n++) {
            const uint32_t row = (uint32_t)min((256 * n + tid) / CH, left);
#pragma unroll
            for (int u = 0; u < 2; u++)
                r[n][u] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, __umul24(row, (uint32_t)pitch) + place.at[n][u], so, 0));
        }
    }
    // Splitting in ten steps a piece, five for either half.
    static constexpr int STEPS = 2 * SplitQuad::STEPS * kN;
    u32x4_t w[3];
    SplitQuad quad;
    float m;
    __device__ __forceinline__ void step(int x, __bf16* buf, int tid, float& chk) {
        const int n = x / (2 * SplitQuad::STEPS), h = x / SplitQuad::STEPS % 2, k = x % SplitQuad::STEPS;
        if (k == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++) quad.r[i] = r[n][h][i];
        }
        uint32_t a = 0, b = 0;
        quad.step(k, a, b);
        if (k % 2 == 0) {
            w[k / 2][2 * h] = a;
            w[k / 2][2 * h + 1] = b;
        }
        if (k == 3) {
            m = split_max(split_max(h == 0 ? 0.0f : m, r[n][h][0]), r[n][h][1]);
            m = split_max(split_max(m, r[n][h][2]), r[n][h][3]);
            asm volatile("" : "+v"(m));  // here: put off behind the next tile's loads, it would keep them out of these registers
        }
        if (h == 1 && k % 2 == 0 && has(n, tid)) {  // a plane at a time: three writes at once hold the wave
            const int idx = 256 * n + tid;
            *(u32x4_t*)(buf + Plane::at(idx / CH, idx % CH) + (k / 2) * Plane::SIZE) = w[k / 2];
        }
        if (h == 1 && k == 4) chk = split_too_small(m) ? kSplitMost : __builtin_fmaxf(chk, m);
    }
    __device__ __forceinline__ void store(__bf16* buf, int tid, float& chk) {
#pragma unroll
        for (int x = 0; x < STEPS; x++) step(x, buf, tid, chk);
    }
    // A operands: chunk j of plane a of row `col`; chunk j of plane a of column 32t + lane % 32
    static __device__ __forceinline__ bf16x8_t row_frag(const __bf16* buf, int a, int j, int col, int hh) {
        return Plane::row_frag(buf + a * Plane::SIZE, j, col, hh);
    }
    static __device__ __forceinline__ bf16x8_t col_frag(const __bf16* buf, int a, int t, int j, int lane) {
        return Plane::col_frag(buf + a * Plane::SIZE, t, j, lane);
    }
};

// The owners' rows: this lane's elements 16j + 8hh .. of row `row` of N rows of D, zeros beyond seq and dim, without a branch, so that
// all are on their way together.
template <int KS>
struct OwnerRow {
    f32x4_t x[KS][2];
    __device__ __forceinline__ void load(const float* src, int row, int N, int D, int hh) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, 4u * (uint32_t)N * (uint32_t)D, kBufferFlags);
        const uint32_t at = row < N ? 4u * (uint32_t)row * (uint32_t)D : 0x80000000u;
#pragma unroll
        for (int j = 0; j < KS; j++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int d = 16 * j + 8 * hh + 4 * u;
                x[j][u] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, d < D ? at + 4u * (uint32_t)d : 0x80000000u, 0, 0));
            }
    }
    __device__ __forceinline__ void split(Split8 (&s)[KS], float& chk) const {
#pragma unroll
        for (int j = 0; j < KS; j++) {
            float y[8];
#pragma unroll
            for (int i = 0; i < 8; i++) y[i] = x[j][i >> 2][i & 3];
            check8(y, chk);
            s[j] = split8(y);
        }
    }
    __device__ __forceinline__ float dot(const OwnerRow& o) const {
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < KS; j++)
#pragma unroll
            for (int i = 0; i < 8; i++) sum = __builtin_fmaf(o.x[j][i >> 2][i & 3], x[j][i >> 2][i & 3], sum);
        return sum;
    }
};

// accumulators (d = 32t + 8g + 4hh + i of row `row`) to row `row` of a [seq, dim] matrix
template <int DT>
__device__ __forceinline__ void store_rows(float* __restrict__ dst, const f32x16_t* acc, int row, int hh, int N, int D) {
    if (row >= N) return;
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d = 32 * t + 8 * g + 4 * hh;
            if (d < D) *(f32x4_t*)(dst + (size_t)row * D + d) = f32x4_t{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
        }
}

__device__ __forceinline__ bf16x8_t as_frag(u32x4_t x) { return __builtin_bit_cast(bf16x8_t, x); }

// (batch, head) and 128-row block of the workgroup at position `lin` of `nt` blocks times `n_bh` pairs: pairs on one XCD each
// where they divide by eight
__device__ __forceinline__ void owner_of_block(int lin, int nt, int n_bh, int& bh, int& blk) {
    const bool by_xcd = (n_bh & 7) == 0;
    const int r = by_xcd ? lin >> 3 : lin;
    bh = r / nt;
    blk = r % nt;
    if (by_xcd) bh = 8 * bh + (lin & 7);
}
__device__ __forceinline__ int linear_block() { return (int)blockIdx.x + (int)gridDim.x * ((int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z); }

// the sum of x over groups of 4 or 8 neighbouring lanes, in each of them
template <int N>
__device__ __forceinline__ float lanes_sum(float x) {
    auto dpp = [](float y, auto ctrl) { return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(y), decltype(ctrl)::value, 0xf, 0xf, true)); };
    x += dpp(x, std::integral_constant<int, 0xb1>{});  // quad_perm 1, 0, 3, 2
    x += dpp(x, std::integral_constant<int, 0x4e>{});  // quad_perm 2, 3, 0, 1
    if (N == 8) x += dpp(x, std::integral_constant<int, 0x141>{});  // row_half_mirror: the other quad
    return x;
}

template <int DT>
constexpr int kLdsHalfs = 4 * Stream<DT>::SIZE;  // two tiles of either streamed matrix

// kOwnDelta: delta is formed here, a tile's with its rows of dO and O, and not read.
template <int DT, bool kOwnDelta>
__device__ __forceinline__ void bwd_dkdv_split(const FlashBwdF32Params& p, int lin, int nt, __bf16* lds, float (*stat)[2][kTile]) {
    constexpr int DPAD = 32 * DT, KS = DPAD / 16;
    using St = Stream<DT>;
    constexpr int BUF = 2 * St::SIZE;  // Q, then dO

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    const int N = p.seq, D = p.dim;
    int bh, blk;
    owner_of_block(lin, nt, p.batch * p.heads, bh, blk);
    const int key = blk * 4 * kTile + wave * kTile + col;
    const size_t base = (size_t)bh * N * D;
    const float* __restrict__ Qg = p.q + base;
    const float* __restrict__ Kg = p.k + base;
    const float* __restrict__ Vg = p.v + base;
    const float* __restrict__ dOg = p.d_out + base;
    const float* __restrict__ lse = p.lse + (size_t)bh * N;
    const float* __restrict__ delta = p.delta + (size_t)bh * N;
    const float* __restrict__ Og = p.o + base;

    float chk = 0.0f;
    Split8 kf[KS], vf[KS];
    {
        OwnerRow<KS> k, v;
        k.load(Kg, key, N, D, hh);
        v.load(Vg, key, N, D, hh);
        k.split(kf, chk);
        v.split(vf, chk);
    }
    // Each sum in two register sets: the large terms (hh), and the five small ones.  The large set is rounded twice a tile
    // instead of twelve times, and no vector instruction touches either.
    f32x16_t acc_dv[DT], acc_dk[DT], low_dv[DT], low_dk[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) {
        zero16(acc_dv[t]);
        zero16(acc_dk[t]);
        zero16(low_dv[t]);
        zero16(low_dk[t]);
    }

    const typename St::Place place(D, tid);
    St q_in(Qg, N, D), o_in(dOg, N, D), out_in(Og, N, D);  // out_in: O, for delta; read and multiplied, never split
    float st = 0.0f;  // threads 0..31: the row statistic, 32..63: delta.  Rows beyond seq: +inf, their weights are zeros
    const float* const st_src = kOwnDelta || lane < 32 ? lse : delta;  // (kOwnDelta: the upper half's is not used)
    auto load = [&](int tile) RT_INLINE {
        q_in.load(tile, place, tid);
        o_in.load(tile, place, tid);
        if constexpr (kOwnDelta) out_in.load(tile, place, tid);
        st = st_src[min(tile * kTile + (lane & 31), N - 1)];  // (in every wave: no branch around a load)
    };
    auto put_delta = [&](int b, int row0) RT_INLINE {  // of the tile's rows of dO and O as they came; returns it
        constexpr int LANES = DPAD / 8;  // of a row
        float x = 0.0f, y = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            x = __builtin_fmaf(o_in.r[0][0][i], out_in.r[0][0][i], x);
            y = __builtin_fmaf(o_in.r[0][1][i], out_in.r[0][1][i], y);
        }
        const int row = tid / LANES;
        x = row0 + row < N ? lanes_sum<LANES>(x + y) : 0.0f;
        if (tid % LANES == 0 && (St::ITEMS % 256 == 0 || tid < St::ITEMS)) stat[b][1][row] = x;
        return x;
    };
    // (the loaded value is looked at here and not where it is requested: there the wave would wait for it)
    auto put_stat = [&](int b, int row0) RT_INLINE {
        if constexpr (kOwnDelta) {
            chk = split_max(chk, put_delta(b, row0));
            if (tid < 32) {
                const bool in = row0 + tid < N;
                chk = split_max(chk, in ? st : 0.0f);
                stat[b][0][tid] = in ? st : -neg_inf();
            }
        } else if (wave == 0) {
            const bool in = row0 + (tid & 31) < N;
            chk = split_max(chk, in ? st : 0.0f);
            stat[b][tid >> 5][tid & 31] = in ? st : (tid < 32 ? -neg_inf() : 0.0f);
        }
    };
    auto store = [&](int b) RT_INLINE {
        q_in.store(lds + b * BUF, tid, chk);
        o_in.store(lds + b * BUF + St::SIZE, tid, chk);
        put_stat(b, 0);
    };
    // P and dS of one pair of elements from the score-shaped products
    auto weight = [&](float s, float dp, float l, float dl, float& pv, float& ds) {
        pv = __builtin_amdgcn_exp2f((s * p.scale - l) * kLog2e);
        ds = pv * (dp - dl) * p.scale;
    };

    const int n_tiles = (N + kTile - 1) / kTile;
    load(0);
    store(0);
    const bool uncarried = __syncthreads_or(!(chk < kSplitMost));  // seen already: no step of the loop below
    load(1);
    // A step's products, in the order S = Q K^T, dP = dO V^T, dV += P^T dO, dK += dS^T Q: no vector work stands alone.  The next tile (in
    // registers since the step before) is split between the instructions of S, P is formed and split between those of dP and
    // the first of dV, dS between those of dV and the first half of dK.  With one wave a SIMD nothing else would keep both
    // units busy.  The scheduling barriers keep that order.
    for (int tile = 0; tile < (uncarried ? 0 : n_tiles); tile++) {
        const __bf16* qb = lds + (tile & 1) * BUF;
        const __bf16* ob = qb + St::SIZE;
        __bf16* nb = lds + ((tile + 1) & 1) * BUF;  // behind the last tile: a repeat that nobody reads
        if constexpr (DT > 1) {
#pragma unroll
            for (int j = 0; j < KS; j++) asm volatile("" : "+a"(kf[j].p[0]), "+a"(kf[j].p[1]), "+a"(kf[j].p[2]), "+a"(vf[j].p[0]), "+a"(vf[j].p[1]), "+a"(vf[j].p[2]));
        }
        f32x16_t s, dp;
        zero16(s);
        zero16(dp);
        bf16x8_t fa[3][KS];
        // S in the order of terms of the forward kernel (there K is the A operand): the same bits, which is what makes
        // exp(S - L) of a dominant key one
        auto read_plane = [&](const __bf16* buf, int a) RT_INLINE {
#pragma unroll
            for (int j = 0; j < KS; j++) fa[a][j] = St::row_frag(buf, a, j, col, hh);
        };
        read_plane(qb, 0);
        f32x4_t lv[4], dl[4];  // register i of S and dP holds query row 8 (i/4) + 4 hh + i%4 of the tile
        u32x4_t pw[2][3], dw[2][3];
        SplitQuad sp;
        float y[4];
        // 16 steps a chunk of P (from S, which becomes P), then 16 a chunk of dS: for four elements at a time the three
        // instructions of each, then their split
        auto weight_step = [&](int x) RT_INLINE {
            const int j = (x / 16) & 1, e = (x / 8) & 1, k = x % 8, i0 = 8 * j + 4 * e, g = i0 >> 2;
            if (k < 3) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (x < 32) {
                        if (k == 0) y[i] = s[i0 + i] * p.scale - lv[g][i];
                        if (k == 1) y[i] *= kLog2e;
                        if (k == 2) sp.r[i] = s[i0 + i] = __builtin_amdgcn_exp2f(y[i]);
                    } else {
                        if (k == 0) y[i] = dp[i0 + i] - dl[g][i];
                        if (k == 1) y[i] *= s[i0 + i];
                        if (k == 2) sp.r[i] = y[i] * p.scale;
                    }
                }
                return;
            }
            uint32_t a = 0, b = 0;
            sp.step(k - 3, a, b);
            if ((k - 3) % 2) return;
            u32x4_t& w = (x < 32 ? pw : dw)[j][(k - 3) / 2];
            w[2 * e] = a;
            w[2 * e + 1] = b;
        };
        auto weights = [&](int from, int to, int n, int of) RT_INLINE {  // the n-th of `of` shares of steps from .. to
#pragma unroll
            for (int x = from + (to - from) * n / of; x < from + (to - from) * (n + 1) / of; x++) weight_step(x);
            RT_ORDER();
        };
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_plane(qb, 1);
            if (n == KS) read_plane(qb, 2);
            s = mfma_h(fa[kTermB[term]][j], kf[j].p[kTermA[term]], s);
#pragma unroll
            for (int x = n * 2 * St::STEPS / (6 * KS); x < (n + 1) * 2 * St::STEPS / (6 * KS); x++) {
                if (x < St::STEPS) q_in.step(x, nb, tid, chk);
                else o_in.step(x - St::STEPS, nb + St::SIZE, tid, chk);
            }
            RT_ORDER();
        }
        put_stat((tile + 1) & 1, (tile + 1) * kTile);  // (behind the last tile: nothing is read there)
        load(tile + 2);  // (behind the last tile: its last row, which nobody reads)
        read_plane(ob, 2);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            lv[g] = *(const f32x4_t*)(&stat[tile & 1][0][8 * g + 4 * hh]);
            dl[g] = *(const f32x4_t*)(&stat[tile & 1][1][8 * g + 4 * hh]);
        }
        bf16x8_t ca[DT][3];
        auto read_cols = [&](const __bf16* buf, int j, int t) RT_INLINE {
#pragma unroll
            for (int a = 0; a < 3; a++) ca[t][a] = St::col_frag(buf, a, t, j, lane);
        };
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_plane(ob, 1);
            if (n == KS) read_plane(ob, 0);
            if (n == 4 * KS) {
#pragma unroll
                for (int t = 0; t < DT; t++) read_cols(ob, 0, t);
            }
            dp = mfma_h(fa[kTermA[term]][j], vf[j].p[kTermB[term]], dp);
            weights(0, 24, n, 6 * KS);
        }
#pragma unroll
        for (int g = 0; g < 2; g++)  // dV, then dK
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int t = 0; t < DT; t++) {
#pragma unroll
                    for (int term = 0; term < 6; term++) {
                        f32x16_t& o = term == 5 ? (g ? acc_dk[t] : acc_dv[t]) : (g ? low_dk[t] : low_dv[t]);
                        o = mfma_h(ca[t][kTermA[term]], as_frag(g ? dw[j][kTermB[term]] : pw[j][kTermB[term]]), o);
                        const int n = 6 * t + term;
                        if (g == 0 && j == 0) weights(24, 36, n, 6 * DT);
                        if (g == 0 && j == 1) weights(36, 48, n, 6 * DT);
                        if (g == 1 && j == 0) weights(48, 64, n, 6 * DT);
                    }
                    if (j == 0) read_cols(g ? qb : ob, 1, t);
                    else if (g == 0) read_cols(qb, 0, t);
                }
        __syncthreads();
    }

#pragma unroll
    for (int t = 0; t < DT; t++) {
        acc_dv[t] += low_dv[t];
        acc_dk[t] += low_dk[t];
    }
    if (uncarried || __syncthreads_or(!(chk < kSplitMost))) {
        // something here the split does not carry: the rows once more in f32, the tiles through LDS two at a time.  For a
        // launch of both kernels (B=4 H=16 N=1024 D=64) 551 us where the first tiles show it, 684 where only the last does;
        // straight from memory 2880; the f32 kernels alone 506.
        using Tile = F32Tile<DT>;
        static_assert(4 * Tile::SIZE * sizeof(float) <= kLdsHalfs<DT> * sizeof(__bf16), "two tiles of Q and dO");
        float* const f32_lds = (float*)lds;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            zero16(acc_dv[t]);
            zero16(acc_dk[t]);
        }
        float k[16 * DT], v[16 * DT];
        f32_row<DT>(k, Kg + (size_t)key * D, key < N, D, hh);
        f32_row<DT>(v, Vg + (size_t)key * D, key < N, D, hh);
        Tile qt, ot;
        float st_f = 0.0f;
        auto load_f = [&](int q0) {
            qt.template load<true>(Qg, (size_t)D, q0, N, D, tid);
            ot.load(dOg, (size_t)D, q0, N, D, tid);
            if constexpr (kOwnDelta) {  // dO once more, as the sum over neighbouring lanes wants it (a row a lane: 409 us, B=1 H=8 N=2048 D=64; this 354)
                o_in.load(q0 / kTile, place, tid);
                out_in.load(q0 / kTile, place, tid);
            }
            if (tid < (kOwnDelta ? 32 : 64)) {
                const int row = q0 + (tid & 31);
                st_f = row < N ? st_src[row] : (tid < 32 ? -neg_inf() : 0.0f);
            }
        };
        auto store_f = [&](int b2, int q0) {
            qt.store(f32_lds + b2 * 2 * Tile::SIZE, tid);
            ot.store(f32_lds + b2 * 2 * Tile::SIZE + Tile::SIZE, tid);
            if constexpr (kOwnDelta) put_delta(b2, q0);
            if (tid < (kOwnDelta ? 32 : 64)) stat[b2][tid >> 5][tid & 31] = st_f;
        };
        load_f(0);
        store_f(0, 0);
        __syncthreads();
        for (int tile = 0; tile < n_tiles; tile++) {
            const float* qb = f32_lds + (tile & 1) * 2 * Tile::SIZE;
            const float* ob = qb + Tile::SIZE;
            if (tile + 1 < n_tiles) load_f((tile + 1) * kTile);
            f32x16_t s, dp;
            zero16(s);
            zero16(dp);
            f32_rows<DT>(s, qb, k, col, hh);
            f32_rows<DT>(dp, ob, v, col, hh);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int r = 8 * (i >> 2) + 4 * hh + (i & 3);
                float pv, ds;
                weight(s[i], dp[i], stat[tile & 1][0][r], stat[tile & 1][1][r], pv, ds);
                s[i] = pv;
                dp[i] = ds;
            }
            f32_cols<DT>(acc_dv, ob, s, col, hh);
            f32_cols<DT>(acc_dk, qb, dp, col, hh);
            if (tile + 1 < n_tiles) store_f((tile + 1) & 1, (tile + 1) * kTile);
            __syncthreads();
        }
    }
    store_rows<DT>(p.dv + base, acc_dv, key, hh, N, D);
    store_rows<DT>(p.dk + base, acc_dk, key, hh, N, D);
}

// kLeaveDelta: for a dK/dV kernel that runs behind this one
template <int DT, bool kLeaveDelta>
__device__ __forceinline__ void bwd_dq_split(const FlashBwdF32Params& p, int lin, int nt, __bf16* lds) {
    constexpr int DPAD = 32 * DT, KS = DPAD / 16;
    using St = Stream<DT>;
    constexpr int BUF = 2 * St::SIZE;  // K, then V

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    const int N = p.seq, D = p.dim;
    int bh, blk;
    owner_of_block(lin, nt, p.batch * p.heads, bh, blk);
    const int q_row = blk * 4 * kTile + wave * kTile + col;
    const bool q_ok = q_row < N;
    const size_t base = (size_t)bh * N * D;
    const float* __restrict__ Qg = p.q + base;
    const float* __restrict__ Kg = p.k + base;
    const float* __restrict__ Vg = p.v + base;
    const float* __restrict__ dOg = p.d_out + base;
    const float* __restrict__ Og = p.o + base;

    // the owner rows, and delta = dO . O of each: half a row in this lane, half in lane + 32
    float chk = 0.0f, delta_q = 0.0f;
    Split8 qf[KS], of[KS];
    {
        OwnerRow<KS> q, g, o;
        q.load(Qg, q_row, N, D, hh);
        g.load(dOg, q_row, N, D, hh);
        o.load(Og, q_row, N, D, hh);
        q.split(qf, chk);
        g.split(of, chk);
        delta_q = g.dot(o);
    }
    delta_q += other_half(delta_q);
    if (kLeaveDelta && hh == 0 && q_ok) p.delta[(size_t)bh * N + q_row] = delta_q;
    float lse_q = q_ok ? p.lse[(size_t)bh * N + q_row] : 0.0f;
    chk = split_max(split_max(chk, lse_q), delta_q);
    if (!q_ok) lse_q = -neg_inf();  // weights of zero

    f32x16_t acc[DT], low[DT];  // as in the kernel above
#pragma unroll
    for (int t = 0; t < DT; t++) {
        zero16(acc[t]);
        zero16(low[t]);
    }
    const typename St::Place place(D, tid);
    St k_in(Kg, N, D), v_in(Vg, N, D);
    auto load = [&](int tile) RT_INLINE {
        k_in.load(tile, place, tid);
        v_in.load(tile, place, tid);
    };
    auto store = [&](int b) {
        k_in.store(lds + b * BUF, tid, chk);
        v_in.store(lds + b * BUF + St::SIZE, tid, chk);
    };
    // dS of one element from the score-shaped products; register i holds key 8 (i/4) + 4 hh + i%4 of the tile
    auto weight = [&](float s, float dp) {
        return __builtin_amdgcn_exp2f((s * p.scale - lse_q) * kLog2e) * (dp - delta_q) * p.scale;
    };
    auto hide_edge = [&](f32x16_t& s, int kv0) {  // keys beyond seq: a score of -inf
        if (kv0 + kTile > N) {
            asm volatile("");  // a branch: the selects cost more than the jump
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (kv0 + 8 * (i >> 2) + 4 * hh + (i & 3) >= N) s[i] = neg_inf();
        }
    };

    const int n_tiles = (N + kTile - 1) / kTile;
    load(0);
    store(0);
    const bool uncarried = __syncthreads_or(!(chk < kSplitMost));  // seen already: no step of the loop below
    load(1);
    for (int tile = 0; tile < (uncarried ? 0 : n_tiles); tile++) {  // a step as in the kernel above, in the order S, dP, dQ
        const __bf16* kb = lds + (tile & 1) * BUF;
        const __bf16* vb = kb + St::SIZE;
        __bf16* nb = lds + ((tile + 1) & 1) * BUF;
        if constexpr (DT > 1) {
#pragma unroll
            for (int j = 0; j < KS; j++) asm volatile("" : "+a"(qf[j].p[0]), "+a"(qf[j].p[1]), "+a"(qf[j].p[2]), "+a"(of[j].p[0]), "+a"(of[j].p[1]), "+a"(of[j].p[2]));
        }
        f32x16_t s, dp;
        zero16(s);
        zero16(dp);
        bf16x8_t fa[2][KS];
        auto read_plane = [&](const __bf16* buf, int a) RT_INLINE {
#pragma unroll
            for (int j = 0; j < KS; j++) fa[a & 1][j] = St::row_frag(buf, a, j, col, hh);
        };
        read_plane(kb, 2);
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_plane(kb, 1);
            if (n == KS) read_plane(kb, 0);
            s = mfma_h(fa[kTermA[term] & 1][j], qf[j].p[kTermB[term]], s);
#pragma unroll
            for (int x = n * 2 * St::STEPS / (6 * KS); x < (n + 1) * 2 * St::STEPS / (6 * KS); x++) {
                if (x < St::STEPS) k_in.step(x, nb, tid, chk);
                else v_in.step(x - St::STEPS, nb + St::SIZE, tid, chk);
            }
            RT_ORDER();
        }
        load(tile + 2);  // (behind the last tile: its last row, which nobody reads)
        read_plane(vb, 2);
        hide_edge(s, tile * kTile);
        u32x4_t dw[2][3];
        SplitQuad sd;
        float y[4];
        // 12 steps of P (S becomes P), then 16 a chunk of dS, four elements at a time as in the kernel above
        auto weight_step = [&](int x) RT_INLINE {
            const int z = x < 12 ? x / 3 : (x - 12) / 8, k = x < 12 ? x % 3 : (x - 12) % 8, i0 = 4 * z;
            if (k < 3) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (x < 12) {
                        if (k == 0) y[i] = s[i0 + i] * p.scale - lse_q;
                        if (k == 1) y[i] *= kLog2e;
                        if (k == 2) s[i0 + i] = __builtin_amdgcn_exp2f(y[i]);
                    } else {
                        if (k == 0) y[i] = dp[i0 + i] - delta_q;
                        if (k == 1) y[i] *= s[i0 + i];
                        if (k == 2) sd.r[i] = y[i] * p.scale;
                    }
                }
                return;
            }
            uint32_t a = 0, b = 0;
            sd.step(k - 3, a, b);
            if ((k - 3) % 2) return;
            u32x4_t& w = dw[z / 2][(k - 3) / 2];
            w[2 * (z & 1)] = a;
            w[2 * (z & 1) + 1] = b;
        };
        auto weights = [&](int from, int to, int n, int of_n) RT_INLINE {
#pragma unroll
            for (int x = from + (to - from) * n / of_n; x < from + (to - from) * (n + 1) / of_n; x++) weight_step(x);
            RT_ORDER();
        };
        bf16x8_t kc[DT][3];
        auto read_cols = [&](int j, int t) RT_INLINE {
#pragma unroll
            for (int a = 0; a < 3; a++) kc[t][a] = St::col_frag(kb, a, t, j, lane);
        };
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_plane(vb, 1);
            if (n == KS) read_plane(vb, 0);
            if (n == 4 * KS) {
#pragma unroll
                for (int t = 0; t < DT; t++) read_cols(0, t);
            }
            dp = mfma_h(fa[kTermA[term] & 1][j], of[j].p[kTermB[term]], dp);
            weights(0, 12, n, 6 * KS);
        }
        weights(12, 28, 0, 1);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int t = 0; t < DT; t++) {
#pragma unroll
                for (int term = 0; term < 6; term++) {
                    f32x16_t& o = term == 5 ? acc[t] : low[t];
                    o = mfma_h(kc[t][kTermA[term]], as_frag(dw[j][kTermB[term]]), o);
                    if (j == 0) weights(28, 44, 6 * t + term, 6 * DT);
                }
                if (j == 0) read_cols(1, t);
            }
        __syncthreads();
    }

#pragma unroll
    for (int t = 0; t < DT; t++) acc[t] += low[t];
    if (uncarried || __syncthreads_or(!(chk < kSplitMost))) {  // as in the kernel above
        using Tile = F32Tile<DT>;
        static_assert(4 * Tile::SIZE * sizeof(float) <= kLdsHalfs<DT> * sizeof(__bf16), "two tiles of K and V");
        float* const f32_lds = (float*)lds;
#pragma unroll
        for (int t = 0; t < DT; t++) zero16(acc[t]);
        float q[16 * DT], o[16 * DT];
        f32_row<DT>(q, Qg + (size_t)q_row * D, q_ok, D, hh);
        f32_row<DT>(o, dOg + (size_t)q_row * D, q_ok, D, hh);
        Tile kt, vt;
        auto load_f = [&](int kv0) {
            kt.load(Kg, (size_t)D, kv0, N, D, tid);
            vt.load(Vg, (size_t)D, kv0, N, D, tid);
        };
        auto store_f = [&](int b2) {
            kt.store(f32_lds + b2 * 2 * Tile::SIZE, tid);
            vt.store(f32_lds + b2 * 2 * Tile::SIZE + Tile::SIZE, tid);
        };
        load_f(0);
        store_f(0);
        __syncthreads();
        for (int tile = 0; tile < n_tiles; tile++) {
            const float* kb = f32_lds + (tile & 1) * 2 * Tile::SIZE;
            if (tile + 1 < n_tiles) load_f((tile + 1) * kTile);
            f32x16_t s, dp;
            zero16(s);
            zero16(dp);
            f32_rows<DT>(s, kb, q, col, hh);
            f32_rows<DT>(dp, kb + Tile::SIZE, o, col, hh);
            hide_edge(s, tile * kTile);
#pragma unroll
            for (int i = 0; i < 16; i++) dp[i] = weight(s[i], dp[i]);
            f32_cols<DT>(acc, kb, dp, col, hh);
            if (tile + 1 < n_tiles) store_f((tile + 1) & 1);
            __syncthreads();
        }
    }
    store_rows<DT>(p.dq + base, acc, q_row, hh, N, D);
}

// One workgroup a CU at head dim 64, so a wave may have the whole register file.
template <int DT>
__global__ __launch_bounds__(256, DT == 1 ? 2 : 1) void flash_bwd_f32_dkdv_split_kernel(FlashBwdF32Params p) {
    __shared__ __attribute__((aligned(16))) __bf16 lds[kLdsHalfs<DT>];
    __shared__ __attribute__((aligned(16))) float stat[2][2][kTile];
    bwd_dkdv_split<DT, false>(p, linear_block(), (int)gridDim.x, lds, stat);
}
template <int DT>
__global__ __launch_bounds__(256, DT == 1 ? 2 : 1) void flash_bwd_f32_dq_split_kernel(FlashBwdF32Params p) {
    __shared__ __attribute__((aligned(16))) __bf16 lds[kLdsHalfs<DT>];
    bwd_dq_split<DT, true>(p, linear_block(), (int)gridDim.x, lds);
}
// Both in one launch, dK/dV, the longer one, first: grid x holds the owner blocks of both.
template <int DT>
__global__ __launch_bounds__(256, DT == 1 ? 2 : 1) void flash_bwd_f32_both_split_kernel(FlashBwdF32Params p) {
    __shared__ __attribute__((aligned(16))) __bf16 lds[kLdsHalfs<DT>];
    __shared__ __attribute__((aligned(16))) float stat[2][2][kTile];
    const int nt = (int)gridDim.x / 2, lin = linear_block(), n = nt * p.batch * p.heads;
    if (lin < n) bwd_dkdv_split<DT, true>(p, lin, nt, lds, stat);
    else bwd_dq_split<DT, false>(p, lin - n, nt, lds);
}

}  // namespace

hipError_t launch_flash_bwd_f32_split(hipStream_t stream, const FlashBwdF32Params& p) {
    dim3 grid((p.seq + 4 * kTile - 1) / (4 * kTile), p.heads, p.batch), block(256);
    const bool both = bwd_f32_one_launch((long long)grid.x * grid.y * grid.z, p.dim <= 32 ? 2 : 1, p.n_cus) && bwd_f32_apart(p);
    auto launch = [&](auto dt_c) {
        constexpr int kDT = decltype(dt_c)::value;
        if (both) {
            hipLaunchKernelGGL(flash_bwd_f32_both_split_kernel<kDT>, dim3(2 * grid.x, grid.y, grid.z), block, 0, stream, p);
            return;
        }
        hipLaunchKernelGGL(flash_bwd_f32_dq_split_kernel<kDT>, grid, block, 0, stream, p);
        hipLaunchKernelGGL(flash_bwd_f32_dkdv_split_kernel<kDT>, grid, block, 0, stream, p);
    };
    if (p.dim <= 32) launch(std::integral_constant<int, 1>{});
    else if (p.dim <= 64) launch(std::integral_constant<int, 2>{});
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace rt

#include "flash_bwd_f32_wide.hpp"
