// Gradients of f32 attention on the bf16 matrix cores, head dims 65 to 128: the split products of flash_bwd_f32_split.hip, 128 owner
// rows a workgroup, where the owners of K and V and the sums of dK and dV together do not fit a wave's registers.  dK and dV are therefore
// workgroups of their own (S is formed once more: eight products instead of seven), and a step is laid out so that every vector
// instruction stands beside a matrix instruction:
//   dP of this tile      beside  P of this tile (its scores were formed in the step before)
//   S of the next tile   beside  dS of this tile and its split
//   the gradient         beside  the split of the tile after the next into LDS
// with one barrier, inside the first product, and everything a product starts with read from LDS in the product ahead of it.  A gradient's
// tile sum is formed in registers of its own, small terms first, and added once (rounded once a tile at its size).
//
// What bounds it: a wave has its SIMD to itself and waits alone.  At head dim 128 a tile of dQ takes 8.4 k clocks, the matrix pipe 4.6 k of them (144
// instructions of 32) and the vector unit 3.1 k; one of dK or dV 7.5 k, 3.8 k and 2.9 k (counters, B=4 H=16 N=1024, clock 2.0 GHz).  us of both gradients, B=4 H=16 N=1024: head dim 128
// f32 kernels 1087, this 863 with sums in the accumulation registers (the vector unit reads none of those), 798 -> 765 with
// them in its own, 740 without copies of loaded registers and owners loaded one behind the other; 96 868, 669, 649, 587.  Relative error
// against 64 bits 6.5e-7 -> 4.2e-7, 6.1e-7 -> 4.1e-7.
// Part of flash_bwd_f32_split.hip, whose helpers it uses.
#pragma once

namespace rt {

namespace {

enum Role { kDQ, kDK, kDV };  // the gradient of a workgroup's rows

// dK and dV: dS and P are split at 2^17 times their size, so that whatever f32 holds of them (2^-126 on) keeps 24 bits.  The last term of a
// split meets the smallest bf16 below 2^-109, and the rows of a key that every query weighs with 2^-123 were off by 2^-12 of themselves, where
// f32 leaves 2^-18 (the exponent's rounding).  (A row of dQ has weights that sum to one, beside which such small ones are nothing.)  dS has
// the factor in its scale, P takes 16 multiplies a tile: training steps, us, without / with, B H N head dim: 1 12 903 96 196.3 / 200.0, 4 8
// 376 80 94.1 / 96.2, 8 16 96 96 49.5 / 50.1, 4 16 453 80 183.0 / 183.7, 2 8 640 128 136.6 / 136.7.  What goes in stays below 2^27 for it:
// 2^(3 x 27 + 7) of a product of three over the head dim, times a scale below 2^-3 and 2^17, is below 2^125 over the 2^23 rows that 2 GiB
// hold.
constexpr float kLift = 0x1p17f, kWideMost = 0x1p27f;

template <int DT>
constexpr int kWideHalfs = 6 * Stream<DT>::SIZE;  // three tiles of either streamed matrix

// X is the matrix the scores are formed with (K for dQ, Q else), Y the one dP is formed with (V, dO); xo and yo the owners' rows.
// kLeaveDelta: dQ leaves delta for a launch that runs behind this one.
template <int DT, Role kRole, bool kLeaveDelta>
__device__ __forceinline__ void bwd_role(const FlashBwdF32Params& p, int lin, int nt, __bf16* lds, float (*stat)[2][kTile]) {
    constexpr bool kQ = kRole == kDQ;   // owners are query rows
    constexpr bool kDP = kRole != kDV;  // has the product dP, and a gradient that contracts over X with dS; dV contracts over Y with P
    constexpr int DPAD = 32 * DT, KS = DPAD / 16;
    constexpr int kAhead = kDP ? 2 : 3;  // tiles X is split ahead of the step
    using St = Stream<DT>;
    using Plane = SplitPlane<DT>;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    const int N = p.seq, D = p.dim;
    int bh, blk;
    owner_of_block(lin, nt, p.batch * p.heads, bh, blk);
    const int row_o = blk * 4 * kTile + wave * kTile + col;
    const bool row_ok = row_o < N;
    const size_t base = (size_t)bh * N * D;
    const float* __restrict__ Xg = (kQ ? p.k : p.q) + base;
    const float* __restrict__ Yg = (kQ ? p.v : p.d_out) + base;
    const float* __restrict__ XOg = (kQ ? p.q : p.k) + base;
    const float* __restrict__ YOg = (kQ ? p.d_out : p.v) + base;
    const float* __restrict__ Og = p.o + base;
    const float* __restrict__ lse = p.lse + (size_t)bh * N;
    const float* __restrict__ delta = p.delta + (size_t)bh * N;

    const typename St::Place place(D, tid);
    St x_in(Xg, N, D), y_in(Yg, N, D);
    float st = 0.0f;  // lanes 0..31: the row statistic, 32..63: delta.  Rows beyond seq: +inf, their weights are zeros
    const float* const st_src = lane < 32 ? lse : delta;
    auto load_y = [&](int tile) RT_INLINE {
        y_in.load(tile, place, tid);
        if (!kQ) st = st_src[min(tile * kTile + (lane & 31), N - 1)];  // (in every wave: no branch around a load)
    };
    x_in.load(0, place, tid);
    load_y(0);

    float chk = 0.0f;
    Split8 xo[KS], yo[KS];
    float lse_q = 0.0f, delta_q = 0.0f;  // kQ: of this lane's row
    {
        OwnerRow<KS> x;
        x.load(XOg, row_o, N, D, hh);
        x.split(xo, chk);
        if constexpr (kDP) {
            x.load(YOg, row_o, N, D, hh);
            x.split(yo, chk);
            if constexpr (kQ) {
                OwnerRow<KS> o;
                o.load(Og, row_o, N, D, hh);
                delta_q = x.dot(o);
            }
        }
    }
    if constexpr (kQ) {
        delta_q += other_half(delta_q);
        if (kLeaveDelta && hh == 0 && row_ok) p.delta[(size_t)bh * N + row_o] = delta_q;
        lse_q = row_ok ? lse[row_o] : 0.0f;
        chk = split_max(split_max(chk, lse_q), delta_q);
        if (!row_ok) lse_q = -neg_inf();  // weights of zero
    }

    f32x16_t acc[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) zero16(acc[t]);
    auto xbuf = [&](int i) RT_INLINE { return lds + i * St::SIZE; };
    auto ybuf = [&](int i) RT_INLINE { return lds + (3 + i) * St::SIZE; };

    // (the loaded value is looked at here and not where it is requested: there the wave would wait for it)
    auto put_stat = [&](int b, int tile) RT_INLINE {
        if (kQ || wave != 0) return;
        const bool in = tile * kTile + (lane & 31) < N;
        chk = split_max(chk, in ? st : 0.0f);
        stat[b][lane >> 5][lane & 31] = in ? st : (lane < 32 ? -neg_inf() : 0.0f);
    };
    auto hide_edge = [&](f32x16_t& s, int kv0) RT_INLINE {  // keys beyond seq: a score of -inf
        if (kQ && kv0 + kTile > N) {
            asm volatile("");  // a branch: the selects cost more than the jump
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (kv0 + 8 * (i >> 2) + 4 * hh + (i & 3) >= N) s[i] = neg_inf();
        }
    };

    // ---- the products.  A score-shaped one is 6 KS instructions, the terms in the order of the forward kernel; plane 2 of the tile
    // is in fa[B] already, plane 1 comes to fa[1 - B] and plane 0 to fa[B] a third ahead of their use.
    bf16x8_t fa[2][KS];
    auto read_plane = [&](const __bf16* buf, int a, int b) RT_INLINE {
#pragma unroll
        for (int j = 0; j < KS; j++) fa[b][j] = Plane::row_frag(buf + a * Plane::SIZE, j, col, hh);
    };
    auto product = [&](f32x16_t& c, const __bf16* buf, const Split8(&own)[KS], int B, auto between) RT_INLINE {
        zero16(c);
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) {
            const int term = n / KS, j = n % KS;
            if (n == 0) read_plane(buf, 1, 1 - B);
            if (n == KS) read_plane(buf, 0, B);
            c = mfma_h(fa[kTermA[term] == 1 ? 1 - B : B][j], own[j].p[kTermB[term]], c);
            between(n);
            RT_ORDER();
        }
    };
    // A gradient: column block t contracted over the tile's 32 rows in registers of its own, the small terms of both halves of the
    // rows ahead of the large ones, then one addition to the sum, made while the next block is multiplied.  The
    // columns of a half are read while the half before it is multiplied.
    bf16x8_t ca[2][3];
    auto read_cols = [&](const __bf16* buf, int t, int j) RT_INLINE {
#pragma unroll
        for (int a = 0; a < 3; a++) ca[j][a] = Plane::col_frag(buf + a * Plane::SIZE, t, j, lane);
    };
    f32x16_t part[2];
    auto gradient = [&](const __bf16* buf, const u32x4_t(&w)[2][3], auto between, auto ahead) RT_INLINE {
#pragma unroll
        for (int t = 0; t < DT; t++) {
            f32x16_t& o = part[t & 1];
            zero16(o);
            bf16x8_t head;
#pragma unroll
            for (int n = 0; n < 12; n++) {
                const int j = n < 10 ? n / 5 : n - 10, term = n < 10 ? n % 5 : 5;
                if (n == 0) read_cols(buf, t, 1);
                if (n == 5) {
                    head = ca[0][0];
                    if (t + 1 < DT) read_cols(buf, t + 1, 0);
                    else ahead();
                }
                o = mfma_h(n == 10 ? head : ca[j][kTermA[term]], as_frag(w[j][kTermB[term]]), o);
                if (t > 0 && n >= 2 && n < 10) {
#pragma unroll
                    for (int i = 2 * (n - 2); i < 2 * (n - 1); i++) {
                        float x = acc[t - 1][i] + part[(t - 1) & 1][i];
                        asm volatile("" : "+v"(x));  // here, and not behind the last block
                        acc[t - 1][i] = x;
                    }
                }
                between(12 * t + n);
                RT_ORDER();
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i++) acc[DT - 1][i] += part[(DT - 1) & 1][i];
    };

    const int n_tiles = (N + kTile - 1) / kTile;
    // tiles 0 and 1 (X: up to kAhead) ahead of the walk
#pragma unroll
    for (int i = 0; i < kAhead; i++) {
        if (i > 0 && i >= n_tiles) break;
        if (i > 0) {
            x_in.load(i, place, tid);
            if (i < 2) load_y(i);
        }
        x_in.store(xbuf(i), tid, chk);
        if (i < 2) {
            put_stat(i, i);
            y_in.store(ybuf(i), tid, chk);
        }
    }
    const bool uncarried = __syncthreads_or(!(chk < kWideMost));  // seen already: no step of the loop below
    f32x16_t s;
    if (!uncarried) {
        x_in.load(kAhead, place, tid);
        load_y(2);
        read_plane(xbuf(0), 2, 1);
        product(s, xbuf(0), xo, 1, [](int) {});
        if constexpr (kDP) read_plane(ybuf(0), 2, 0);
        else if (n_tiles > 1) read_plane(xbuf(1), 2, 1);
    }
    // A step: dP of this tile beside its P; the scores of the next tile beside this tile's dS; the gradients beside the split of
    // the tile after the next.  Its one barrier, a third into the first product, stands between the writes of the step before and
    // the first read of what they wrote, and between the last reads of the tile before and the writes over it.
    const float ds_scale = kQ ? p.scale : p.scale * kLift;
    int b0 = 0;  // tile % 3
    for (int tile = 0; tile < (uncarried ? 0 : n_tiles); tile++) {
        const int b1 = b0 == 2 ? 0 : b0 + 1, b2 = b1 == 2 ? 0 : b1 + 1;
        const bool more = tile + 1 < n_tiles;
        if constexpr (DT > 1) {
#pragma unroll
            for (int j = 0; j < KS; j++) {
                asm volatile("" : "+a"(xo[j].p[0]), "+a"(xo[j].p[1]), "+a"(xo[j].p[2]));
                if constexpr (kDP) asm volatile("" : "+a"(yo[j].p[0]), "+a"(yo[j].p[1]), "+a"(yo[j].p[2]));
            }
        }
        hide_edge(s, tile * kTile);
        f32x4_t lv[4], dl[4];  // register i of S and dP holds row 8 (i/4) + 4 hh + i%4 of the tile
        if constexpr (!kQ) {
#pragma unroll
            for (int g = 0; g < 4; g++) lv[g] = *(const f32x4_t*)(&stat[b0][0][8 * g + 4 * hh]);
        }
        u32x4_t w[2][3];  // dS, or P where dV contracts over it
        SplitQuad sq;
        float y[4];
        f32x16_t dp, s_next;
        // eight steps for four elements, of P (dV) nine: the three instructions of each, the factor of P in a step of its own (one behind the
        // exponentials it waits for them, 1 x 12 heads of 96, N=903 201 us for 196), then the five of their split
        constexpr int kPSteps = 9;
        auto split_part = [&](int z, int k) RT_INLINE {
            uint32_t a = 0, b = 0;
            sq.step(k, a, b);
            if (k % 2) return;
            w[z / 2][k / 2][2 * (z & 1)] = a;
            w[z / 2][k / 2][2 * (z & 1) + 1] = b;
        };
        auto p_part = [&](int z, int k) RT_INLINE {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (k == 0) y[i] = s[4 * z + i] * p.scale - (kQ ? lse_q : lv[z][i]);
                if (k == 1) y[i] *= kLog2e;
                if (k == 2) s[4 * z + i] = __builtin_amdgcn_exp2f(y[i]);
                if (k == 3) sq.r[i] = s[4 * z + i] * kLift;
            }
        };
        auto p_step = [&](int x) RT_INLINE {
            const int z = x / kPSteps, k = x % kPSteps;
            if (k < 4) p_part(z, k);
            else split_part(z, k - 4);
        };
        auto ds_step = [&](int x) RT_INLINE {
            const int z = x / 8, k = x % 8;
            if (k >= 3) return split_part(z, k - 3);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (k == 0) y[i] = dp[4 * z + i] - (kQ ? delta_q : dl[z][i]);
                if (k == 1) y[i] *= s[4 * z + i];
                if (k == 2) sq.r[i] = y[i] * ds_scale;
            }
        };
        auto shares = [&](auto step, int steps, int n, int of) RT_INLINE {  // the n-th of `of` shares
#pragma unroll
            for (int x = steps * n / of; x < steps * (n + 1) / of; x++) step(x);
        };
        auto p_only = [&](int x) RT_INLINE { p_part(x / 3, x % 3); };  // P without its split
        if constexpr (kDP) {
            product(dp, ybuf(b0), yo, 0, [&](int n) RT_INLINE {
                if (n == 2 * KS - 1) __syncthreads();
                shares(p_only, 12, n, 6 * KS);
                if (n == 4 * KS) read_plane(xbuf(b1), 2, 1);
            });
            if constexpr (!kQ) {
#pragma unroll
                for (int g = 0; g < 4; g++) dl[g] = *(const f32x4_t*)(&stat[b0][1][8 * g + 4 * hh]);
            }
            if (more) {
                product(s_next, xbuf(b1), xo, 1, [&](int n) RT_INLINE {
                    shares(ds_step, 32, n, 6 * KS);
                    if (n == 5 * KS) read_cols(xbuf(b0), 0, 0);
                });
            } else {
                zero16(s_next);
                shares(ds_step, 32, 0, 1);
                read_cols(xbuf(b0), 0, 0);
            }
        } else {
            if (more) {
                product(s_next, xbuf(b1), xo, 1, [&](int n) RT_INLINE {
                    if (n == 2 * KS - 1) __syncthreads();
                    shares(p_step, 4 * kPSteps, n, 6 * KS);
                    if (n == 5 * KS) read_cols(ybuf(b0), 0, 0);
                });
            } else {
                zero16(s_next);
                __syncthreads();
                shares(p_step, 4 * kPSteps, 0, 1);
                read_cols(ybuf(b0), 0, 0);
            }
        }
        __bf16* const xn = xbuf(kAhead == 2 ? b2 : b0);
        auto feed = [&](int n) RT_INLINE {
            constexpr int kAll = 2 * St::STEPS;
#pragma unroll
            for (int x = kAll * n / (12 * DT); x < kAll * (n + 1) / (12 * DT); x++) {
                if (x == 0) put_stat(b2, tile + 2);
                if (x < St::STEPS) y_in.step(x, ybuf(b2), tid, chk);
                else x_in.step(x - St::STEPS, xn, tid, chk);
            }
        };
        gradient(kDP ? xbuf(b0) : ybuf(b0), w, feed, [&]() RT_INLINE {  // and what the next step reads first
            if constexpr (kDP) read_plane(ybuf(b1), 2, 0);
            else read_plane(xbuf(b2), 2, 1);
        });
        x_in.load(tile + kAhead + 1, place, tid);  // behind the last tile: its last row, read by nobody
        load_y(tile + 3);
        s = s_next;
        b0 = b1;
    }

    if constexpr (!kQ) {
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[t][i] *= 1.0f / kLift;
    }

    if (uncarried || __syncthreads_or(!(chk < kWideMost))) {
        // something here the split does not carry: the rows once more in f32, the tiles through LDS two at a time
        using Tile = F32Tile<DT>;
        static_assert(4 * Tile::SIZE * sizeof(float) <= kWideHalfs<DT> * sizeof(__bf16), "two tiles of either matrix");
        float* const f32_lds = (float*)lds;
#pragma unroll
        for (int t = 0; t < DT; t++) zero16(acc[t]);
        float x[16 * DT], y[16 * DT];
        f32_row<DT>(x, XOg + (size_t)row_o * D, row_ok, D, hh);
        f32_row<DT>(y, YOg + (size_t)row_o * D, kDP && row_ok, D, hh);
        Tile xt, yt;
        float st_f = 0.0f;
        auto load_f = [&](int tile) RT_INLINE {
            const int row0 = tile * kTile;
            xt.template load<!kQ>(Xg, (size_t)D, row0, N, D, tid);
            yt.load(Yg, (size_t)D, row0, N, D, tid);
            if (!kQ && tid < 64) {
                const int row = row0 + (tid & 31);
                st_f = row < N ? st_src[row] : (tid < 32 ? -neg_inf() : 0.0f);
            }
        };
        auto store_f = [&](int b) RT_INLINE {
            xt.store(f32_lds + b * 2 * Tile::SIZE, tid);
            yt.store(f32_lds + b * 2 * Tile::SIZE + Tile::SIZE, tid);
            if (!kQ && tid < 64) stat[b][tid >> 5][tid & 31] = st_f;
        };
        load_f(0);
        store_f(0);
        __syncthreads();
        for (int tile = 0; tile < n_tiles; tile++) {
            const float* xb = f32_lds + (tile & 1) * 2 * Tile::SIZE;
            const float* yb = xb + Tile::SIZE;
            if (tile + 1 < n_tiles) load_f(tile + 1);
            f32x16_t sf, dp;
            zero16(sf);
            zero16(dp);
            f32_rows<DT>(sf, xb, x, col, hh);
            if constexpr (kDP) f32_rows<DT>(dp, yb, y, col, hh);
            hide_edge(sf, tile * kTile);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int r = 8 * (i >> 2) + 4 * hh + (i & 3);
                const float pv = __builtin_amdgcn_exp2f((sf[i] * p.scale - (kQ ? lse_q : stat[tile & 1][0][r])) * kLog2e);
                dp[i] = pv * (dp[i] - (kQ ? delta_q : stat[tile & 1][1][r])) * p.scale;
                sf[i] = pv;
            }
            if constexpr (kDP) f32_cols<DT>(acc, xb, dp, col, hh);
            else f32_cols<DT>(acc, yb, sf, col, hh);
            if (tile + 1 < n_tiles) store_f((tile + 1) & 1);
            __syncthreads();
        }
    }
    store_rows<DT>((kQ ? p.dq : kDP ? p.dk : p.dv) + base, acc, row_o, hh, N, D);
}

template <int DT>
__global__ __launch_bounds__(256, 1) void flash_bwd_f32_dq_wide_kernel(FlashBwdF32Params p) {
    __shared__ __attribute__((aligned(16))) __bf16 lds[kWideHalfs<DT>];
    bwd_role<DT, kDQ, true>(p, linear_block(), (int)gridDim.x, lds, nullptr);
}
// dK and dV; with kAll dQ as well, between them: the longer ones first.  Grid x holds the owner blocks of each.
template <int DT, bool kAll>
__global__ __launch_bounds__(256, 1) void flash_bwd_f32_dkdv_wide_kernel(FlashBwdF32Params p) {
    __shared__ __attribute__((aligned(16))) __bf16 lds[kWideHalfs<DT>];
    __shared__ __attribute__((aligned(16))) float stat[3][2][kTile];
    const int nt = (int)gridDim.x / (kAll ? 3 : 2), lin = linear_block(), n = nt * p.batch * p.heads;
    if (lin < n) bwd_role<DT, kDK, false>(p, lin, nt, lds, stat);
    else if (kAll && lin < 2 * n) bwd_role<DT, kDQ, false>(p, lin - n, nt, lds, nullptr);
    else bwd_role<DT, kDV, false>(p, lin - (kAll ? 2 * n : n), nt, lds, stat);
}

// delta = dO . O of each row ahead of a launch of all three; half a wave a row
__global__ __launch_bounds__(256) void flash_bwd_f32_delta_kernel(FlashBwdF32Params p) {
    const size_t row = (size_t)blockIdx.x * 8 + (threadIdx.x >> 5), rows = (size_t)p.batch * p.heads * p.seq;
    const int d = 4 * (threadIdx.x & 31);
    float x = 0.0f;
    if (row < rows && d < p.dim) {
        const f32x4_t a = *(const f32x4_t*)(p.d_out + row * p.dim + d), b = *(const f32x4_t*)(p.o + row * p.dim + d);
#pragma unroll
        for (int i = 0; i < 4; i++) x = __builtin_fmaf(a[i], b[i], x);
    }
#pragma unroll
    for (int off = 16; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
    if (row < rows && (threadIdx.x & 31) == 0) p.delta[row] = x;
}

}  // namespace

hipError_t launch_flash_bwd_f32_wide(hipStream_t stream, const FlashBwdF32Params& p) {
    dim3 grid((p.seq + 4 * kTile - 1) / (4 * kTile), p.heads, p.batch), block(256);
    const long long n = (long long)grid.x * grid.y * grid.z;
    const bool all = n < (p.n_cus > 0 ? p.n_cus : 256);
    auto launch = [&](auto dt_c) {
        constexpr int kDT = decltype(dt_c)::value;
        if (all) {
            const size_t rows = (size_t)p.batch * p.heads * p.seq;
            hipLaunchKernelGGL(flash_bwd_f32_delta_kernel, dim3((unsigned)((rows + 7) / 8)), block, 0, stream, p);
            hipLaunchKernelGGL((flash_bwd_f32_dkdv_wide_kernel<kDT, true>), dim3(3 * grid.x, grid.y, grid.z), block, 0, stream, p);
            return;
        }
        hipLaunchKernelGGL(flash_bwd_f32_dq_wide_kernel<kDT>, grid, block, 0, stream, p);
        hipLaunchKernelGGL((flash_bwd_f32_dkdv_wide_kernel<kDT, false>), dim3(2 * grid.x, grid.y, grid.z), block, 0, stream, p);
    };
    if (p.dim <= 64) return hipErrorInvalidValue;
    else if (p.dim <= 96) launch(std::integral_constant<int, 3>{});
    else if (p.dim <= 128) launch(std::integral_constant<int, 4>{});
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace rt
