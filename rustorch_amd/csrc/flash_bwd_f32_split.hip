// Gradients of f32 attention on the bf16 matrix cores, every operand as three bf16 terms (rt_split.hpp): the two kernels of
// flash_bwd_f32.hip (its header has the formulas) for launches with enough rows to fill the chip with 128 a workgroup.
//
// A wave owns 32 rows (keys for dK/dV, queries for dQ), split once into registers as B operands; the four waves of a
// workgroup walk the same tiles of 32 rows of the other side, which the workgroup splits into LDS: as rows (A operand of the
// score-shaped products) and, where a gradient contracts over them, as columns (A operand of dV^T += dO^T P and the like,
// the rows of a column in the order the weights sit in the accumulators).  Every output row has one owner: no atomics, the
// same bits on every launch.
//
// What bounds them: matrix and vector instructions together, as in the forward kernel (counted: 38 % and 43 % of the clocks of
// either kernel); at head dim 64 a tile is 72 (dQ) and 96 (dK/dV) matrix instructions of 32 clocks and about 580 and 745
// vector ones of 4 per wave.  LDS holds two tiles of both streams for one workgroup a CU, and a wave takes the register
// file of its SIMD; the moves that makes necessary are a tenth of the vector instructions.  Between two matrix instructions stands a
// step of the next tile's split or of the weights (two matrix instructions behind each other hold the wave until the first
// is done: 382 -> 370 us; without any order 418).  B=4 H=16 N=1024 D=64, dQ and dK/dV: 506 -> 370 us, B=2 N=2048 973 ->
// 704, head dim 32 273 -> 216; relative error against 64 bits 5.9e-7 -> 4.5e-7, 7.3e-7 -> 5.9e-7, 5.5e-7 -> 4.4e-7.
#include "rt_common.hpp"
#include "rt_kernels.hpp"
#include "rt_split.hpp"

namespace rt {

namespace {

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

// One streamed matrix [N, D]: a tile's rows and columns on their way from memory into LDS.  Rows behind the last repeat it;
// whoever reads the tile gives them weights of zero.
template <int DT, bool kRowsOut, bool kColsOut>
struct Stream {
    static constexpr int DPAD = 32 * DT, LDK = DPAD + 8, LDV = kTile + 8;
    static constexpr int RPL = kTile * LDK, CPL = DPAD * LDV;
    static constexpr int SIZE = (kRowsOut ? 3 * RPL : 0) + (kColsOut ? 3 * CPL : 0);  // bf16 elements of a tile
    static constexpr int COLS = kRowsOut ? 3 * RPL : 0;                               // where its columns begin
    static constexpr int ITEMS = 4 * DPAD;
    f32x4_t r[2];
    float c[8];

    __device__ __forceinline__ void clear() {
        r[0] = r[1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 8; e++) c[e] = 0.0f;
    }
    __device__ __forceinline__ void load(const float* __restrict__ src, int row0, int N, int D, int tid) {
        if (ITEMS % 256 != 0 && tid >= ITEMS) return;
        if constexpr (kRowsOut) {
            const int row = min(row0 + tid / (DPAD / 8), N - 1), d = 8 * (tid % (DPAD / 8));
            const float* x = src + (size_t)row * D + d;
#pragma unroll
            for (int u = 0; u < 2; u++) {
                f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
                if (d + 4 * u < D) z = *(const f32x4_t*)(x + 4 * u);
                r[u] = z;
            }
        }
        if constexpr (kColsOut) {
            const int d = tid % DPAD, g = tid / DPAD;
            const int first = row0 + 16 * (g >> 1) + 4 * (g & 1);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int row = min(first + 8 * (e >> 2) + (e & 3), N - 1);
                c[e] = d < D ? src[(size_t)row * D + d] : 0.0f;
            }
        }
    }
    // Splitting in twelve steps a row (or column) piece of eight elements: step x is term x % 3 of pair x / 3, the last writes.
    u32x4_t w[3];
    SplitPair pair;
    float m;
    template <bool kCol>
    __device__ __forceinline__ void step(int x, __bf16* buf, int tid, float& chk) {
        const int e = x / 3, n = x % 3;
        if (n == 0) pair.r = kCol ? split_f32x2_t{c[2 * e], c[2 * e + 1]} : split_f32x2_t{r[e >> 1][2 * (e & 1)], r[e >> 1][2 * (e & 1) + 1]};
        w[n][e] = pair.step(n);
        if (!kCol && n == 2) {  // the columns hold the same values
            const float x0 = r[e >> 1][2 * (e & 1)], x1 = r[e >> 1][2 * (e & 1) + 1];
            if (e == 0) m = 0.0f;
            m = split_max(split_max(m, x0), x1);
            if (e == 3) chk = split_too_small(m) ? kSplitMost : __builtin_fmaxf(chk, m);
        }
        if (x == 11 && (ITEMS % 256 == 0 || tid < ITEMS)) {
            __bf16* at = kCol ? buf + COLS + (tid % DPAD) * LDV + 8 * (tid / DPAD)
                              : buf + (tid / (DPAD / 8)) * LDK + 8 * (tid % (DPAD / 8));
#pragma unroll
            for (int u = 0; u < 3; u++) *(u32x4_t*)(at + u * (kCol ? CPL : RPL)) = w[u];
        }
    }
    __device__ __forceinline__ void store(__bf16* buf, int tid, float& chk) {
#pragma unroll
        for (int x = 0; x < 12; x++)
            if constexpr (kRowsOut) step<false>(x, buf, tid, chk);
#pragma unroll
        for (int x = 0; x < 12; x++)
            if constexpr (kColsOut) step<true>(x, buf, tid, chk);
    }
    // A operands: chunk j of plane a of row `col`; slots 16j + 8hh .. of plane a of column 32t + col
    static __device__ __forceinline__ bf16x8_t row_frag(const __bf16* buf, int a, int j, int col, int hh) {
        return *(const bf16x8_t*)(buf + a * RPL + col * LDK + 16 * j + 8 * hh);
    }
    static __device__ __forceinline__ bf16x8_t col_frag(const __bf16* buf, int a, int t, int j, int col, int hh) {
        return *(const bf16x8_t*)(buf + COLS + a * CPL + (32 * t + col) * LDV + 16 * j + 8 * hh);
    }
};

// 8 elements of a row, zeros beyond seq and dim
__device__ __forceinline__ void load8(float (&x)[8], const float* __restrict__ src, int row, int d, int N, int D) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
        f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
        if (row < N && d + 4 * u < D) z = *(const f32x4_t*)(src + (size_t)row * D + d + 4 * u);
#pragma unroll
        for (int i = 0; i < 4; i++) x[4 * u + i] = z[i];
    }
}

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

// (batch, head) and 128-row block of a workgroup: pairs on one XCD each where they divide by eight
__device__ __forceinline__ void owner_of_block(int& bh, int& blk) {
    const int nt = (int)gridDim.x, n_bh = (int)(gridDim.y * gridDim.z);
    bh = (int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z;
    blk = (int)blockIdx.x;
    if ((n_bh & 7) == 0) {
        const int lin = (int)blockIdx.x + nt * bh, xcd = lin & 7, r = lin >> 3;
        bh = (r / nt) * 8 + xcd;
        blk = r % nt;
    }
}

// Two tiles of both streams in LDS (117 KB at head dim 64): one workgroup a CU, so a wave may have the whole register file.
template <int DT>
__global__ __launch_bounds__(256, DT == 1 ? 2 : 1) void flash_bwd_f32_dkdv_split_kernel(FlashBwdF32Params p) {
    constexpr int DPAD = 32 * DT, KS = DPAD / 16;
    using St = Stream<DT, true, true>;
    constexpr int BUF = 2 * St::SIZE;  // Q, then dO
    __shared__ __attribute__((aligned(16))) __bf16 lds[2 * BUF];
    __shared__ __attribute__((aligned(16))) float stat[2][2][kTile];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, hh = lane >> 5;
    const int N = p.seq, D = p.dim;
    int bh, blk;
    owner_of_block(bh, blk);
    const int key = blk * 4 * kTile + wave * kTile + col;
    const size_t base = (size_t)bh * N * D;
    const float* __restrict__ Qg = p.q + base;
    const float* __restrict__ Kg = p.k + base;
    const float* __restrict__ Vg = p.v + base;
    const float* __restrict__ dOg = p.d_out + base;
    const float* __restrict__ lse = p.lse + (size_t)bh * N;
    const float* __restrict__ delta = p.delta + (size_t)bh * N;

    float chk = 0.0f;
    Split8 kf[KS], vf[KS];
#pragma unroll
    for (int j = 0; j < KS; j++) {
        float x[8];
        load8(x, Kg, key, 16 * j + 8 * hh, N, D);
        check8(x, chk);
        kf[j] = split8(x);
        load8(x, Vg, key, 16 * j + 8 * hh, N, D);
        check8(x, chk);
        vf[j] = split8(x);
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

    St q_in, o_in;
    q_in.clear();
    o_in.clear();
    float st = 0.0f;  // threads 0..31: the row statistic, 32..63: delta.  Rows beyond seq: +inf, their weights are zeros
    auto load = [&](int row0) {
        q_in.load(Qg, row0, N, D, tid);
        o_in.load(dOg, row0, N, D, tid);
        if (tid < 64) {
            const int row = row0 + (tid & 31);
            st = row < N ? (tid < 32 ? lse : delta)[row] : 0.0f;
            chk = split_max(chk, st);
            if (row >= N && tid < 32) st = -neg_inf();
        }
    };
    auto store = [&](int b) {
        q_in.store(lds + b * BUF, tid, chk);
        o_in.store(lds + b * BUF + St::SIZE, tid, chk);
        if (tid < 64) stat[b][tid >> 5][tid & 31] = st;
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
    if (n_tiles > 1) load(kTile);
    // In a step the next tile (in registers since the step before) is split between the instructions of the score-shaped
    // products, and the second half of the weights is formed between those of the first half's gradient products: with one
    // wave a SIMD nothing else would keep both units busy.  The scheduling barriers keep that order.
    for (int tile = 0; tile < (uncarried ? 0 : n_tiles); tile++) {
        const __bf16* qb = lds + (tile & 1) * BUF;
        const __bf16* ob = qb + St::SIZE;
        __bf16* nb = lds + ((tile + 1) & 1) * BUF;  // behind the last tile: a repeat that nobody reads
        f32x16_t s, dp;
        zero16(s);
        zero16(dp);
        bf16x8_t qa[3][KS], oa[2][KS];
        // S in the order of terms of the forward kernel (there K is the A operand): the same bits, which is what makes
        // exp(S - L) of a dominant key one
        auto read_q = [&](int a) {
#pragma unroll
            for (int j = 0; j < KS; j++) qa[a][j] = St::row_frag(qb, a, j, col, hh);
        };
        auto read_o = [&](int a) {
#pragma unroll
            for (int j = 0; j < KS; j++) oa[a & 1][j] = St::row_frag(ob, a, j, col, hh);
        };
        read_q(0);
        read_o(2);
        auto stage = [&](int n) {  // behind instruction n of 12 KS: its share of the 48 steps of the next tile's split
#pragma unroll
            for (int x = n * 48 / (12 * KS); x < (n + 1) * 48 / (12 * KS); x++) {
                St& in = x < 24 ? q_in : o_in;
                __bf16* to = nb + (x < 24 ? 0 : St::SIZE);
                if ((x % 24) < 12) in.template step<false>(x % 12, to, tid, chk);
                else in.template step<true>(x % 12, to, tid, chk);
            }
            RT_ORDER();
        };
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_q(1), read_o(1);
            if (n == KS) read_q(2), read_o(0);
            s = mfma_h(qa[kTermB[term]][j], kf[j].p[kTermA[term]], s);
            stage(2 * n);
            dp = mfma_h(oa[kTermA[term] & 1][j], vf[j].p[kTermB[term]], dp);
            stage(2 * n + 1);
        }
        if (tid < 64) stat[(tile + 1) & 1][tid >> 5][tid & 31] = st;
        if (tile + 2 < n_tiles) load((tile + 2) * kTile);
        // register i holds query row 8 (i/4) + 4 hh + i%4 of the tile
        f32x4_t lv[4], dl[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            lv[g] = *(const f32x4_t*)(&stat[tile & 1][0][8 * g + 4 * hh]);
            dl[g] = *(const f32x4_t*)(&stat[tile & 1][1][8 * g + 4 * hh]);
        }
        u32x4_t pw[2][3], dw[2][3];
        SplitPair sp, sd;
        auto weight_step = [&](int j, int x) {  // 24 steps a chunk, six a pair
            const int e = x / 6, n = x % 6, i = 8 * j + 2 * e;
            if (n < 2) {
                float pv, ds;
                weight(s[i + n], dp[i + n], lv[i >> 2][(i & 3) + n], dl[i >> 2][(i & 3) + n], pv, ds);
                sp.r[n] = pv;
                sd.r[n] = ds;
            } else if (n == 2) {
                pw[j][0][e] = sp.step(0);
            } else if (n == 3) {
                pw[j][1][e] = sp.step(1);
            } else if (n == 4) {
                pw[j][2][e] = sp.step(2);
                dw[j][0][e] = sd.step(0);
            } else {
                dw[j][1][e] = sd.step(1);
                dw[j][2][e] = sd.step(2);
            }
        };
        bf16x8_t oc[DT][3], qc[DT][3];
        auto read_cols = [&](int j, int t) {
#pragma unroll
            for (int a = 0; a < 3; a++) {
                oc[t][a] = St::col_frag(ob, a, t, j, col, hh);
                qc[t][a] = St::col_frag(qb, a, t, j, col, hh);
            }
        };
#pragma unroll
        for (int t = 0; t < DT; t++) read_cols(0, t);
#pragma unroll
        for (int x = 0; x < 24; x++) weight_step(0, x);
        RT_ORDER();
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int t = 0; t < DT; t++) {
#pragma unroll
                for (int term = 0; term < 6; term++) {
                    const int n = 6 * t + term;
                    auto form = [&](int n2) {  // behind instruction n2 of 12 DT: its share of the second chunk's weights
                        if (j == 1) return;
#pragma unroll
                        for (int x = n2 * 24 / (12 * DT); x < (n2 + 1) * 24 / (12 * DT); x++) weight_step(1, x);
                        RT_ORDER();
                    };
                    f32x16_t& ov = term == 5 ? acc_dv[t] : low_dv[t];
                    f32x16_t& ok = term == 5 ? acc_dk[t] : low_dk[t];
                    ov = mfma_h(oc[t][kTermA[term]], as_frag(pw[j][kTermB[term]]), ov);
                    form(2 * n);
                    ok = mfma_h(qc[t][kTermA[term]], as_frag(dw[j][kTermB[term]]), ok);
                    form(2 * n + 1);
                }
                if (j == 0) read_cols(1, t);
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
        static_assert(4 * Tile::SIZE * sizeof(float) <= sizeof(lds), "two tiles of Q and dO");
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
            qt.load(Qg, (size_t)D, q0, N, D, tid);
            ot.load(dOg, (size_t)D, q0, N, D, tid);
            if (tid < 64) {
                const int row = q0 + (tid & 31);
                st_f = row < N ? (tid < 32 ? lse : delta)[row] : (tid < 32 ? -neg_inf() : 0.0f);
            }
        };
        auto store_f = [&](int b2) {
            qt.store(f32_lds + b2 * 2 * Tile::SIZE, tid);
            ot.store(f32_lds + b2 * 2 * Tile::SIZE + Tile::SIZE, tid);
            if (tid < 64) stat[b2][tid >> 5][tid & 31] = st_f;
        };
        load_f(0);
        store_f(0);
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
            if (tile + 1 < n_tiles) store_f((tile + 1) & 1);
            __syncthreads();
        }
    }
    store_rows<DT>(p.dv + base, acc_dv, key, hh, N, D);
    store_rows<DT>(p.dk + base, acc_dk, key, hh, N, D);
}

template <int DT>
__global__ __launch_bounds__(256, DT == 1 ? 2 : 1) void flash_bwd_f32_dq_split_kernel(FlashBwdF32Params p) {
    constexpr int DPAD = 32 * DT, KS = DPAD / 16;
    using StK = Stream<DT, true, true>;
    using StV = Stream<DT, true, false>;
    constexpr int BUF = StK::SIZE + StV::SIZE;
    __shared__ __attribute__((aligned(16))) __bf16 lds[2 * BUF];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, hh = lane >> 5;
    const int N = p.seq, D = p.dim;
    int bh, blk;
    owner_of_block(bh, blk);
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
#pragma unroll
    for (int j = 0; j < KS; j++) {
        float x[8], y[8];
        load8(x, Qg, q_row, 16 * j + 8 * hh, N, D);
        check8(x, chk);
        qf[j] = split8(x);
        load8(x, dOg, q_row, 16 * j + 8 * hh, N, D);
        check8(x, chk);
        of[j] = split8(x);
        load8(y, Og, q_row, 16 * j + 8 * hh, N, D);
#pragma unroll
        for (int i = 0; i < 8; i++) delta_q = __builtin_fmaf(y[i], x[i], delta_q);
    }
    delta_q += other_half(delta_q);
    if (hh == 0 && q_ok) p.delta[(size_t)bh * N + q_row] = delta_q;
    float lse_q = q_ok ? p.lse[(size_t)bh * N + q_row] : 0.0f;
    chk = split_max(split_max(chk, lse_q), delta_q);
    if (!q_ok) lse_q = -neg_inf();  // weights of zero

    f32x16_t acc[DT], low[DT];  // as in the kernel above
#pragma unroll
    for (int t = 0; t < DT; t++) {
        zero16(acc[t]);
        zero16(low[t]);
    }
    StK k_in;
    StV v_in;
    k_in.clear();
    v_in.clear();
    auto load = [&](int row0) {
        k_in.load(Kg, row0, N, D, tid);
        v_in.load(Vg, row0, N, D, tid);
    };
    auto store = [&](int b) {
        k_in.store(lds + b * BUF, tid, chk);
        v_in.store(lds + b * BUF + StK::SIZE, tid, chk);
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
    if (n_tiles > 1) load(kTile);
    for (int tile = 0; tile < (uncarried ? 0 : n_tiles); tile++) {  // a step as in the kernel above
        const __bf16* kb = lds + (tile & 1) * BUF;
        const __bf16* vb = kb + StK::SIZE;
        __bf16* nb = lds + ((tile + 1) & 1) * BUF;
        f32x16_t s, dp;
        zero16(s);
        zero16(dp);
        bf16x8_t ka[2][KS], va[2][KS];
        auto read_rows = [&](int a) {
#pragma unroll
            for (int j = 0; j < KS; j++) {
                ka[a & 1][j] = StK::row_frag(kb, a, j, col, hh);
                va[a & 1][j] = StV::row_frag(vb, a, j, col, hh);
            }
        };
        read_rows(2);
        auto stage = [&](int n) {  // behind instruction n of 12 KS: its share of the 36 steps of the next tile's split
#pragma unroll
            for (int x = n * 36 / (12 * KS); x < (n + 1) * 36 / (12 * KS); x++) {
                if (x < 12) k_in.template step<false>(x % 12, nb, tid, chk);
                else if (x < 24) k_in.template step<true>(x % 12, nb, tid, chk);
                else v_in.template step<false>(x % 12, nb + StK::SIZE, tid, chk);
            }
            RT_ORDER();
        };
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_rows(1);
            if (n == KS) read_rows(0);
            s = mfma_h(ka[kTermA[term] & 1][j], qf[j].p[kTermB[term]], s);
            stage(2 * n);
            dp = mfma_h(va[kTermA[term] & 1][j], of[j].p[kTermB[term]], dp);
            stage(2 * n + 1);
        }
        if (tile + 2 < n_tiles) load((tile + 2) * kTile);
        hide_edge(s, tile * kTile);
        u32x4_t dw[2][3];
        bf16x8_t kc[DT][3];
        auto read_cols = [&](int j, int t) {
#pragma unroll
            for (int a = 0; a < 3; a++) kc[t][a] = StK::col_frag(kb, a, t, j, col, hh);
        };
        SplitPair sd;
        auto weight_step = [&](int j, int x) {  // 12 steps a chunk, three a pair
            const int e = x / 3, n = x % 3, i = 8 * j + 2 * e;
            if (n < 2) {
                sd.r[n] = weight(s[i + n], dp[i + n]);
            } else {
#pragma unroll
                for (int u = 0; u < 3; u++) dw[j][u][e] = sd.step(u);
            }
        };
#pragma unroll
        for (int t = 0; t < DT; t++) read_cols(0, t);
#pragma unroll
        for (int x = 0; x < 12; x++) weight_step(0, x);
        RT_ORDER();
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int t = 0; t < DT; t++) {
#pragma unroll
                for (int term = 0; term < 6; term++) {
                    const int n = 6 * t + term;
                    f32x16_t& o = term == 5 ? acc[t] : low[t];
                    o = mfma_h(kc[t][kTermA[term]], as_frag(dw[j][kTermB[term]]), o);
                    if (j == 0) {
#pragma unroll
                        for (int x = n * 12 / (6 * DT); x < (n + 1) * 12 / (6 * DT); x++) weight_step(1, x);
                        RT_ORDER();
                    }
                }
                if (j == 0) read_cols(1, t);
            }
        __syncthreads();
    }

#pragma unroll
    for (int t = 0; t < DT; t++) acc[t] += low[t];
    if (uncarried || __syncthreads_or(!(chk < kSplitMost))) {  // as in the kernel above
        using Tile = F32Tile<DT>;
        static_assert(4 * Tile::SIZE * sizeof(float) <= sizeof(lds), "two tiles of K and V");
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

}  // namespace

hipError_t launch_flash_bwd_f32_split(hipStream_t stream, const FlashBwdF32Params& p) {
    dim3 grid((p.seq + 4 * kTile - 1) / (4 * kTile), p.heads, p.batch), block(256);
    if (p.dim <= 32) {
        hipLaunchKernelGGL(flash_bwd_f32_dq_split_kernel<1>, grid, block, 0, stream, p);
        hipLaunchKernelGGL(flash_bwd_f32_dkdv_split_kernel<1>, grid, block, 0, stream, p);
    } else if (p.dim <= 64) {
        hipLaunchKernelGGL(flash_bwd_f32_dq_split_kernel<2>, grid, block, 0, stream, p);
        hipLaunchKernelGGL(flash_bwd_f32_dkdv_split_kernel<2>, grid, block, 0, stream, p);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace rt
