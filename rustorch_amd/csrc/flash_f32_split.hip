// f32 flash-attention forward on the bf16 matrix cores, every operand as three bf16 terms (rt_split.hpp).
//
// A workgroup of four waves owns 128 query rows, 32 a wave; all four walk the same key tiles of 32, which the workgroup
// splits once and keeps in LDS as three planes of rows of K (the A operand of S^T = K Q^T) and three of V, read as columns by
// the transposing reads (the A operand of O^T = V^T P^T, the keys of a column in the order the weights sit in the score
// accumulators).  Q is split once into registers, the weights where they are formed.
//
// What bounds it: matrix and vector instructions together.  A tile of 32 keys is 48 matrix instructions of 32 clocks and
// about 370 vector instructions of 4 per wave (1.5 us a tile on a SIMD, with one wave or two); 64 matrix instructions of 64
// clocks in the f32 kernel.  The vector steps are runs of independent instructions between the matrix instructions
// (SplitQuad).  B=4 H=16 N=1024 D=64: f32 kernel 181 us, V loaded and split by columns 99.3, by rows 96.4; causal 120, 67.1,
// 65.4; B=2 N=2048 336, 187.8, 183.6; 5 x 16 heads N=777 D=80 unmasked 229 -> 202.  Above head dim 64 a wave has its SIMD to
// itself: Q in the accumulation registers, D=128 f32 405, 212, 201 us, causal 249, 126, 118.5.  Relative error against 64 bits
// 4.2e-7 -> 1.7e-7 and 5.1e-7 -> 2.2e-7 at the first and third size (four instructions round a score at its size instead of
// 32, one addition a tile the output instead of 16).
#include <type_traits>

#include "rt_common.hpp"
#include "rt_kernels.hpp"
#include "rt_split.hpp"

namespace rt {

namespace {

#define RT_INLINE __attribute__((always_inline))  // lambdas over the wave's registers: a call would put them in memory

constexpr int kTile = 32;  // keys per step, query rows per wave

template <int DT, bool kExactD, bool kCausal>
__global__ __launch_bounds__(256, DT <= 2 ? 2 : 1) void flash_fwd_f32_split_kernel(FlashF32Params p) {
    constexpr int DPAD = 32 * DT;
    constexpr int KS = DPAD / 16;          // contraction chunks of the score product
    using Plane = SplitPlane<DT>;
    constexpr int BUF = 3 * Plane::SIZE;   // a tile of K or of V
    constexpr int ITEMS = 4 * DPAD;        // groups of 8 elements of a tile of K (or V)
    constexpr int NI = (ITEMS + 255) / 256;
    // tiles t and t + 1 of K, t to t + 2 of V
    __shared__ __attribute__((aligned(16))) __bf16 lds[5 * BUF];

    // the arguments, requested together: left to itself the compiler loads a field where it is first used, and waits for it there
    asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.out), "s"(p.lse), "s"(p.heads), "s"(p.group), "s"(p.seq), "s"(p.seq_kv), "s"(p.dim), "s"(p.scale),
                 "s"(p.zigzag), "s"(p.dealt), "s"(p.blocks_magic), "s"(p.heads_magic), "s"(p.lq.batch_stride), "s"(p.lq.head_stride), "s"(p.lq.row_pitch));
    asm volatile("" ::"s"(p.lkv.batch_stride), "s"(p.lkv.head_stride), "s"(p.lkv.row_pitch), "s"(p.lo.batch_stride), "s"(p.lo.head_stride), "s"(p.lo.row_pitch));
    const int Nq = p.seq, N = p.seq_kv ? p.seq_kv : p.seq;
    const int D = kExactD ? DPAD : p.dim;
    // p.zigzag 2 (head dims above 64): a workgroup takes two blocks of a head, a long and a short one, in turn
    const int nq = (int)gridDim.x, n_bh = (int)(gridDim.y * gridDim.z), n_blk = (Nq + 4 * kTile - 1) / (4 * kTile);
    int h = blockIdx.y, b = blockIdx.z;
    int x = (int)blockIdx.x;
    bool short_first = false;
    if (p.dealt) {                        // a head's workgroups on one XCD: its K and V come into one L2
        const int lin = (int)blockIdx.x + nq * ((int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z);
        const int xcd = lin & 7, r = lin >> 3, half = (nq * (n_bh >> 3)) >> 1;
        const int at = div_magic(r, p.blocks_magic), bh = at * 8 + xcd;
        x = r - at * nq;
        // all resident at once: list positions r and r + half share a CU, a long one and a short one of them
        short_first = p.zigzag == 1 && r >= half && div_magic(half, p.blocks_magic) * nq == half;
        b = div_magic(bh, p.heads_magic);
        h = bh - b * (int)gridDim.y;
    }
    int qblk = short_first ? x : n_blk - 1 - x;  // longest causal rows first
    const int kvh = p.group == 1 ? h : h / p.group;
    const float* __restrict__ Qg = p.q + (size_t)b * p.lq.batch_stride + (size_t)h * p.lq.head_stride;
    const float* __restrict__ Kg = p.k + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    const float* __restrict__ Vg = p.v + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    float* __restrict__ Og = p.out + (size_t)b * p.lo.batch_stride + (size_t)h * p.lo.head_stride;
    const size_t q_pitch = p.lq.row_pitch, kv_pitch = p.lkv.row_pitch, o_pitch = p.lo.row_pitch;

    for (;;) {
        int tid = threadIdx.x;
        if constexpr (DT > 2 && kCausal) asm volatile("" : "+v"(tid));  // formed once a block, not kept in registers between two
        const int lane = tid & 63, wave = tid >> 6;
        const int col = lane & 31, hh = lane >> 5;
        const int q0 = qblk * 4 * kTile, q0w = q0 + wave * kTile;
        const int q_row = q0w + col;
        float chk = 0.0f;  // the largest magnitude of everything this thread splits
        uint32_t v_least = ~0u;  // the smallest magnitude of what it splits of V, zeros left out: 2 (bits of |x|) - 1

        // Q as B operand: chunk j, this lane's 8 elements d = 16j + 8hh ..
        // (rows behind the last repeat it, so that no load stands behind a test; nothing of theirs is written)
        const float* const q_at = Qg + (size_t)min(q_row, Nq - 1) * q_pitch;
        Split8 qf[KS];
#pragma unroll
        for (int j = 0; j < KS; j++) {
            float x[8];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int d = 16 * j + 8 * hh + 4 * u;
                f32x4_t z = *(const f32x4_t*)(q_at + (kExactD ? d : min(d, D - 4)));
                if (!kExactD && d >= D) z = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 4; i++) x[4 * u + i] = z[i];
            }
#pragma unroll
            for (int i = 0; i < 8; i++) chk = split_max(chk, x[i]);
            qf[j] = split8(x);
        }

        f32x16_t acc_o[DT];
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc_o[t][i] = 0.0f;
        float m_run = neg_inf(), l_run = 0.0f, l_low = 0.0f;  // l_low: what the additions to l_run rounded off

        const int kv_end = kCausal ? min(N, q0 + 4 * kTile) : N;
        const int n_tiles = (kv_end + kTile - 1) / kTile;
        const int wave_end = q0w >= Nq ? 0 : (kCausal ? min(N, q0w + kTile) : N);
        const int n_wave = (wave_end + kTile - 1) / kTile;  // tiles this wave has scores in

        // A tile's way into LDS: 8 elements of a row per item, of K and of V.  Rows behind the last key repeat
        // it: their weights are exact zeros, and what a zero makes of its value the key itself has made of every row.
        f32x4_t kreg[NI][2], vreg[NI][2];
        uint32_t at[NI];  // byte offsets of this thread's items from a tile's first row
#pragma unroll
        for (int n = 0; n < NI; n++) {  // threads without an item split zeros
            kreg[n][0] = kreg[n][1] = vreg[n][0] = vreg[n][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            const int idx = 256 * n + tid;
            at[n] = 4u * ((uint32_t)(idx / (DPAD / 8)) * (uint32_t)kv_pitch + 8u * (uint32_t)(idx % (DPAD / 8)));
        }
        auto load_tile = [&](int tile) RT_INLINE {
            const bool inside = tile * kTile + kTile <= N;  // wave-uniform
            const char* kb = (const char*)(Kg + (size_t)tile * kTile * kv_pitch);
            const char* vb = (const char*)(Vg + (size_t)tile * kTile * kv_pitch);
#pragma unroll
            for (int n = 0; n < NI; n++) {
                const int idx = 256 * n + tid, d = 8 * (idx % (DPAD / 8));
                if (ITEMS % 256 == 0 || idx < ITEMS) {
                    const size_t off = inside ? (size_t)at[n] : 4 * ((size_t)(min(tile * kTile + idx / (DPAD / 8), N - 1) - tile * kTile) * kv_pitch + (size_t)d);
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f}, y = z;
                        if (kExactD || d + 4 * u < D) {
                            z = *(const f32x4_t*)(kb + off + 16 * u);
                            y = *(const f32x4_t*)(vb + off + 16 * u);
                        }
                        kreg[n][u] = z;
                        vreg[n][u] = y;
                    }
                }
            }
        };
        // Splitting: 20 NI steps, five (SplitQuad) for each half of this thread's K and V items; a plane is written as soon as
        // both halves have given their part of it.
        constexpr int kSplits = 4 * SplitQuad::STEPS * NI;
        SplitQuad quad;
        u32x4_t w[3];
        auto split_step = [&](int x, __bf16* kbuf, __bf16* vbuf) RT_INLINE {
            const int k = x % SplitQuad::STEPS, y = x / SplitQuad::STEPS, h = y & 1, n = y >> 2;
            const bool is_v = (y & 2) != 0;
            const f32x4_t& in = is_v ? vreg[n][h] : kreg[n][h];
            if (k == 0) {
#pragma unroll
                for (int i = 0; i < 4; i++) quad.r[i] = in[i];
            }
            uint32_t a = 0, b = 0;
            quad.step(k, a, b);
            if (k % 2 == 0) {
                w[k / 2][2 * h] = a;
                w[k / 2][2 * h + 1] = b;
            } else if (k == 1) {
                chk = split_max(split_max(chk, in[0]), in[1]);
                chk = split_max(split_max(chk, in[2]), in[3]);
            } else if (is_v) {  // scores of small keys are small whatever is lost of them; small values are the result's size
#pragma unroll
                for (int i = 0; i < 4; i++) v_least = min(v_least, (__float_as_uint(in[i]) << 1) - 1u);
            }
            const int idx = 256 * n + tid;
            if (h == 1 && k % 2 == 0 && (ITEMS % 256 == 0 || idx < ITEMS))
                *(u32x4_t*)((is_v ? vbuf : kbuf) + Plane::at(idx / (DPAD / 8), idx % (DPAD / 8)) + (k / 2) * Plane::SIZE) = w[k / 2];
        };
        auto store_tile = [&](__bf16* kbuf, __bf16* vbuf) RT_INLINE {
#pragma unroll
            for (int x = 0; x < kSplits; x++) split_step(x, kbuf, vbuf);
        };
        auto carried = [&]() RT_INLINE { return chk < kSplitMost && v_least >= kSplitLeast; };
        // of this lane's results: one that is no larger than what a small value of V may have lost of itself
        auto small_result = [&]() RT_INLINE {
            const float least = (l_run + other_half(l_run)) * kSplitLeastResult;
            bool small = false;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (kExactD || 32 * t + 8 * (i >> 2) + 4 * hh + (i & 3) < D) small |= __builtin_fabsf(acc_o[t][i]) < least;
            return small && q_row < Nq;
        };

        // A score tile (register i: key 8 (i/4) + 4 hh + i%4, query `col`): masked, then turned into weights.  The maximum is
        // scaled, the scores are where it is subtracted.
        auto hide = [&](f32x16_t& s, int kv0) RT_INLINE {
            if ((kv0 + kTile > N) || (kCausal && kv0 + kTile - 1 > q0w)) {
                asm volatile("");  // a branch: the selects cost more than the jump
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int kr = kv0 + 8 * (i >> 2) + 4 * hh + (i & 3);
                    if (kr >= N || (kCausal && kr > q_row)) s[i] = neg_inf();
                }
            }
        };
        auto row_max = [&](const f32x16_t& s) RT_INLINE {
            float m_tile = neg_inf();  // NaN never wins, as in the reference's `if x > m`
#pragma unroll
            for (int i = 0; i < 16; i++) m_tile = __builtin_fmaxf(m_tile, s[i]);
            auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(m_tile), __float_as_uint(m_tile), false, false);
            return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * p.scale;
        };
        // the maximum goes to m_run; returns what is subtracted from the scores
        float alpha = 0.0f;
        auto take_max = [&](float m_tile) RT_INLINE {
            const float m_new = __builtin_fmaxf(m_tile, m_run);
            const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
            alpha = (m_run == neg_inf()) ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_use) * kLog2e);
            m_run = m_new;
            return m_use;
        };
        auto add_sum = [&](float tile_l) RT_INLINE {
            const float add = tile_l - l_low * alpha, before = l_run * alpha;
            l_run = before + add;
            l_low = (l_run - before) - add;
        };
        auto rescale = [&]() RT_INLINE {
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int t = 0; t < DT; t++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc_o[t][i] *= alpha;
            }
        };
        // The 6 KS instructions of a score product: planes (a, c) of the six terms, the small ones first.  A plane of K is
        // read from LDS one plane ahead of its use.
        constexpr int kPlaneA[6] = {2, 1, 1, 0, 0, 0}, kPlaneC[6] = {0, 1, 0, 2, 1, 0};
        bf16x8_t kf[2][KS];
        auto read_plane = [&](const __bf16* kbuf, int a) RT_INLINE {
#pragma unroll
            for (int j = 0; j < KS; j++) kf[a & 1][j] = Plane::row_frag(kbuf + a * Plane::SIZE, j, col, hh);
        };
        auto score_step = [&](const __bf16* kbuf, f32x16_t& s, int n) RT_INLINE {  // n: 0 .. 6 KS - 1, a constant
            const int term = n / KS, j = n % KS;
            if (n == 0) read_plane(kbuf, 1);
            if (n == KS) read_plane(kbuf, 0);  // plane 2 has been used
            s = mfma_h(kf[kPlaneA[term] & 1][j], qf[j].p[kPlaneC[term]], s);
        };
        auto zero16 = [](f32x16_t& x) RT_INLINE {
#pragma unroll
            for (int i = 0; i < 16; i++) x[i] = 0.0f;
        };

        __bf16* const v_lds = lds + 2 * BUF;
        load_tile(0);
        store_tile(lds, v_lds);
        if (n_tiles > 1) {
            load_tile(1);
            store_tile(lds + BUF, v_lds + BUF);
        }
        // Seen already: no step of the loop below, straight to the second pass, whose first tile may overwrite what a late
        // wave still reads here for scores that nobody uses then.  (Small values of V alone: only where the tile split last has no
        // others.)
        bool uncarried = __syncthreads_or(!carried());
        if (uncarried) {
            float v_most = 0.0f;
#pragma unroll
            for (int n = 0; n < NI; n++)
#pragma unroll
                for (int i = 0; i < 8; i++) v_most = split_max(v_most, vreg[n][i >> 2][i & 3]);
            uncarried = __syncthreads_or(!(chk < kSplitMost)) || !__syncthreads_or(v_most >= kSplitLeastResult);
        }
        f32x16_t s_next;
        zero16(s_next);
        read_plane(lds, 2);
#pragma unroll
        for (int n = 0; n < 6 * KS; n++) score_step(lds, s_next, n);
        int v_now = 0;  // tile % 3
        // A step multiplies the next tile's scores while this tile's weights are formed, and this tile's weights with V while
        // the tile after the next is split: the matrix instructions have vector work between them in the same wave.  The
        // scheduling barriers keep that order; left to itself the compiler puts the one kind behind the other.
        for (int tile = 0; tile < (uncarried ? 0 : n_tiles); tile++) {
            const __bf16* kn = lds + ((tile + 1) & 1) * BUF;  // behind the last tile: scores of no tile, not used
            const __bf16* vb = v_lds + v_now * BUF;
            if constexpr (DT > 2) {  // what only matrix instructions read goes to the accumulation registers (the sums too: 222 us for 201)
#pragma unroll
                for (int j = 0; j < KS; j++) asm volatile("" : "+a"(qf[j].p[0]), "+a"(qf[j].p[1]), "+a"(qf[j].p[2]));
            }
            if (tile + 2 < n_tiles) load_tile(tile + 2);
            f32x16_t s = s_next;
            hide(s, tile * kTile);
            read_plane(kn, 2);
            zero16(s_next);
            // a third of the score product beside the row maximum, the rest beside the weights, two at a time
#pragma unroll
            for (int n = 0; n < 2 * KS; n++) score_step(kn, s_next, n);
            const float m_use = take_max(row_max(s));
            rescale();
            u32x4_t pw[2][3];
            float part[2] = {0.0f, 0.0f};
            SplitQuad sp;
            float y[4];
            auto weight_step = [&](int x) RT_INLINE {  // 32 steps: four weights at a time, the three instructions of each, their split
                const int g = x / 8, k = x % 8;
                if (k < 3) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if (k == 0) y[i] = __builtin_fmaf(s[4 * g + i], p.scale, -m_use);
                        if (k == 1) y[i] *= kLog2e;
                        if (k == 2) sp.r[i] = __builtin_amdgcn_exp2f(y[i]);
                    }
                    if (k == 2) {
#pragma unroll
                        for (int i = 0; i < 4; i++) part[i & 1] += sp.r[i];
                    }
                    return;
                }
                uint32_t a = 0, b = 0;
                sp.step(k - 3, a, b);
                if ((k - 3) % 2) return;
                pw[g >> 1][(k - 3) / 2][2 * (g & 1)] = a;
                pw[g >> 1][(k - 3) / 2][2 * (g & 1) + 1] = b;
            };
            RT_ORDER();
#pragma unroll
            for (int n = 0; n < 4 * KS; n++) {
                score_step(kn, s_next, 2 * KS + n);
#pragma unroll
                for (int x = n * 32 / (4 * KS); x < (n + 1) * 32 / (4 * KS); x++) weight_step(x);
                RT_ORDER();
            }
            add_sum(part[0] + part[1]);
            // A tile's product in registers of its own, smallest terms first, then one addition to the sum: in the sum
            // itself each of the twelve instructions would round at its size, and the error against 64 bits grew above
            // that of the f32 kernel.
            __bf16* const k_put = lds + (tile & 1) * BUF;
            __bf16* const v_put = v_lds + (v_now == 0 ? 2 : v_now - 1) * BUF;  // tile + 2's
#pragma unroll
            for (int t = 0; t < DT; t++) {
                f32x16_t o;
                zero16(o);
                bf16x8_t v[3][2];
#pragma unroll
                for (int a = 2; a >= 0; a--)
#pragma unroll
                    for (int j = 0; j < 2; j++) v[a][j] = Plane::col_frag(vb + a * Plane::SIZE, t, j, lane);
#pragma unroll
                for (int term = 0; term < 6; term++) {
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        o = mfma_h(v[kPlaneA[term]][j], __builtin_bit_cast(bf16x8_t, pw[j][kPlaneC[term]]), o);
                        // its share of the next tile's split, behind 12 DT instructions
                        const int n = (6 * t + term) * 2 + j;
#pragma unroll
                        for (int x = n * kSplits / (12 * DT); x < (n + 1) * kSplits / (12 * DT); x++) split_step(x, k_put, v_put);
                        RT_ORDER();
                    }
                }
#pragma unroll
                for (int i = 0; i < 16; i++) acc_o[t][i] += o[i];
            }
            v_now = v_now == 2 ? 0 : v_now + 1;
            __syncthreads();
        }

        if (uncarried || (__syncthreads_or(!carried()) && __syncthreads_or(!(chk < kSplitMost) || small_result()))) {
            // something here the split does not carry: the rows once more in f32, the tiles through LDS two at a time.  For a
            // launch (B=4 H=16 N=1024 D=64) 158 us where the first tiles show it, 240 where only the last does; straight from
            // memory 770; the f32 kernel alone 181.
            using Tile = F32Tile<DT>;
            static_assert(4 * Tile::SIZE * sizeof(float) <= sizeof(lds), "two tiles of K and V");
            float* const f32_lds = (float*)lds;
            int tid_f = tid;  // what follows from it is formed here, not kept in registers through the loop above
            asm volatile("" : "+v"(tid_f));
            const int col_f = tid_f & 31, hh_f = (tid_f >> 5) & 1;
#pragma unroll
            for (int t = 0; t < DT; t++) zero16(acc_o[t]);
            m_run = neg_inf();
            l_run = l_low = 0.0f;
            float q[16 * DT];
            f32_row<DT>(q, Qg + (size_t)q_row * q_pitch, q_row < Nq, D, hh_f);
            Tile kt, vt;
            auto load = [&](int tile) RT_INLINE {
                kt.load(Kg, kv_pitch, tile * kTile, N, D, tid_f);
                vt.load(Vg, kv_pitch, tile * kTile, N, D, tid_f);
            };
            auto store = [&](int tile) RT_INLINE {
                kt.store(f32_lds + (tile & 1) * 2 * Tile::SIZE, tid_f);
                vt.store(f32_lds + (tile & 1) * 2 * Tile::SIZE + Tile::SIZE, tid_f);
            };
            load(0);
            store(0);
            __syncthreads();
            for (int tile = 0; tile < n_tiles; tile++) {
                const float* kb = f32_lds + (tile & 1) * 2 * Tile::SIZE;
                if (tile + 1 < n_tiles) load(tile + 1);
                if (tile < n_wave) {
                    f32x16_t s;
                    zero16(s);
                    f32_rows<DT>(s, kb, q, col_f, hh_f);
                    hide(s, tile * kTile);
                    const float m_use = take_max(row_max(s));
                    float tile_l = 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], p.scale, -m_use) * kLog2e);
                        tile_l += s[i];
                    }
                    add_sum(tile_l);
                    rescale();
                    f32_cols<DT>(acc_o, kb + Tile::SIZE, s, col_f, hh_f);
                }
                if (tile + 1 < n_tiles) store(tile + 1);
                __syncthreads();
            }
        }

        const float l = l_run + other_half(l_run);
        const bool good = (l > 0.0f) && (fabsf(l) != __uint_as_float(0x7f800000u)) && (l == l);
        const float inv_l = 1.0f / l;
        if (q_row < Nq) {
        if (p.lse && hh == 0) p.lse[((size_t)b * p.heads + h) * (size_t)Nq + q_row] = m_run + logf(l);
        float* o_row = Og + (size_t)q_row * o_pitch;
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d = 32 * t + 8 * g + 4 * hh;
                f32x4_t o;
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = good ? acc_o[t][4 * g + i] * inv_l : quiet_nan();
                if (kExactD || d < D) *(f32x4_t*)(o_row + d) = o;
            }
        }
        // (every wave is behind a barrier behind its last tile: those of the next block may come into LDS)
        if (DT <= 2 || !kCausal || p.zigzag != 2 || qblk == x || n_blk - 1 - x == x) return;
        qblk = x;
    }
}

// The same products for launches with few rows: a workgroup owns 32 query rows and its four waves share the keys, wave w
// tiles w, w + 4, ..; each walks alone, without a barrier, and the four (O, m, l) are folded through LDS at the end, as in
// flash_fwd_f32_splitk_kernel.  A wave's tile of K and its tile of V lie in LDS of its own as they are in memory (16-byte
// slots of a row XORed with bits of the row), brought there straight; K is requested again once its scores are formed, V
// once it has been multiplied.  Every wave splits what it reads itself, between the matrix instructions of the piece before.
//
// What bounds it: the vector unit, with two workgroups a CU up to head dim 64 and one above (a wave then has its SIMD to itself, Q in
// the accumulation registers): at head dim 64 about 700 instructions a tile and wave, half of them splits of K
// and V that a workgroup of 128 rows shares.  us, f32 kernel -> this, B H N head dim: causal 1 8 2048 64 52.5 -> 42.6, 2 12 999 64
// 46.0 -> 36.8, 1 4 3664 32 63.6 -> 45.9, 1 8 3438 128 271 -> 213, 1 12 1500 96 109 -> 79, 2 4 333 68 17.7 -> 15.5; unmasked 1 8 1024 64
// 28.5 -> 23.2, 1 8 512 64 15.6 -> 13.1, 1 8 1024 96 39.7 -> 29.9; 1 8 2048 64 90.2 -> 68.7 (from 128 rows a workgroup).  Eight waves that
// share them, one workgroup a CU: 1 8 2048 64 42.6 -> 42.8, 4096 128 -> 140, unmasked 1 4 1024 22.2 -> 20.2, not kept.  Relative error
// against 64 bits at head dim 128, N = 2048 unmasked 5.8e-7 -> 2.0e-7.
template <int DT, bool kExactD, bool kCausal>
__global__ __launch_bounds__(256, DT <= 2 ? 2 : 1) void flash_fwd_f32_split_keys_kernel(FlashF32Params p) {
    constexpr int DPAD = 32 * DT, KS = DPAD / 16, SL = DPAD / 4, NREQ = 4 * DT, ROWB = DPAD * 4;
    constexpr int TILE = 32 * DPAD;  // floats
    constexpr int NW = 4, LDO = DPAD + 4;
    __shared__ __attribute__((aligned(1024))) float lds[NW * 2 * TILE];
    __shared__ float red_m[NW][kTile], red_l[NW][kTile], fin_inv[kTile];
    static_assert(2 * TILE >= 32 * LDO, "a wave's partial O fits over its tiles");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    const int Nq = p.seq, N = p.seq_kv ? p.seq_kv : p.seq;
    const int D = kExactD ? DPAD : p.dim;
    // (batch, head) and query tile as in flash_fwd_f32_splitk_kernel: a head's tiles on one XCD, and where all workgroups
    // are resident at once a long and a short one on a CU
    const int nq = (int)gridDim.x, n_bh = (int)(gridDim.y * gridDim.z);
    int h = blockIdx.y, b = blockIdx.z;
    int qtile = nq - 1 - (int)blockIdx.x;
    if (p.dealt) {
        const int lin = (int)blockIdx.x + nq * ((int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z);
        const int xcd = lin & 7, r = lin >> 3, half = (nq * (n_bh >> 3)) >> 1;
        const int at = div_magic(r, p.blocks_magic), bh = at * 8 + xcd;
        qtile = nq - 1 - (r - at * nq);
        if (p.zigzag && r >= half && (div_magic(half, p.blocks_magic) * nq == half || nq == 2 * half)) qtile = (r - half) - div_magic(r - half, p.blocks_magic) * nq;
        b = div_magic(bh, p.heads_magic);
        h = bh - b * (int)gridDim.y;
    } else if (p.zigzag && ((h + b * (int)gridDim.y) * 2 >= n_bh)) {
        qtile = (int)blockIdx.x;
    }
    const int q0 = qtile * kTile, q_row = q0 + col;
    const int kvh = p.group == 1 ? h : h / p.group;
    const float* __restrict__ Qg = p.q + (size_t)b * p.lq.batch_stride + (size_t)h * p.lq.head_stride;
    const float* __restrict__ Kg = p.k + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    const float* __restrict__ Vg = p.v + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    float* __restrict__ Og = p.out + (size_t)b * p.lo.batch_stride + (size_t)h * p.lo.head_stride;
    const size_t q_pitch = p.lq.row_pitch, o_pitch = p.lo.row_pitch;

    const int kv_end = kCausal ? min(N, q0 + kTile) : N;
    const int n_tiles = (kv_end + kTile - 1) / kTile;

    // ---- a wave's tiles: instruction n brings chunks 64 n .. + 63 of 16 bytes, chunk c slot c % SL of row c / SL
    auto swizzle = [](int r) RT_INLINE { return DT % 2 == 0 ? (r & 15) : ((r >> 1) & 7); };
    unsigned char* const Kw = (unsigned char*)(lds + wave * 2 * TILE);
    unsigned char* const Vw = Kw + TILE * 4;
    const uint32_t k_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)Kw, v_lds = k_lds + TILE * 4;
    const uint32_t pitch_b = (uint32_t)p.lkv.row_pitch * 4u;
    uint32_t lane_off[NREQ];
    uint64_t on[NREQ];
#pragma unroll
    for (int n = 0; n < NREQ; n++) {
        const int c = 64 * n + lane, row = c / SL, slot = (c % SL) ^ swizzle(row);
        lane_off[n] = (uint32_t)row * pitch_b + 16u * (uint32_t)slot;
        on[n] = kExactD ? ~0ull : __ballot(4 * slot < D);
        if (!kExactD && 4 * slot >= D) *(u32x4_t*)(Kw + 16 * c) = *(u32x4_t*)(Vw + 16 * c) = u32x4_t{0u, 0u, 0u, 0u};
    }
    const uint32_t kv_bytes = (uint32_t)(N - 1) * pitch_b + 4u * (uint32_t)D;
    const u32x4_t k_rsrc = make_rsrc(Kg, kv_bytes), v_rsrc = make_rsrc(Vg, kv_bytes);
    // (rows behind the last are zeros: their scores are masked, and their weights are zeros.  Tiles behind the last, whose
    // offset lies past the descriptor's end, bring zeros too, without a read, but are requested all the same, so that a wait
    // can count.)
    auto request = [&](const u32x4_t& rs, uint32_t at, int tile) RT_INLINE {
        const uint32_t off = (uint32_t)tile * (uint32_t)kTile * pitch_b;
#pragma unroll
        for (int n = 0; n < NREQ; n++) buffer_to_lds_of(on[n], rs, lane_off[n], off, at + 1024u * (uint32_t)n);
    };
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    request(k_rsrc, k_lds, wave);
    request(v_rsrc, v_lds, wave);

    // ---- operands out of LDS
    const uint32_t k_base = (uint32_t)(col * ROWB + (((2 * hh) ^ swizzle(col)) * 16));
    auto read_k = [&](int j, float (&x)[8]) RT_INLINE {  // elements 16j + 8hh .. of key `col`
#pragma unroll
        for (int u = 0; u < 2; u++) {
            // (rows of 24 slots, DT 3: only the lower three bits of a slot are XORed)
            const uint32_t at = DT == 3 ? (k_base ^ (uint32_t)((4 * (j & 1) + u) * 16)) + (uint32_t)(128 * (j >> 1)) : k_base ^ (uint32_t)((4 * j + u) * 16);
            const f32x4_t z = *(const f32x4_t*)(Kw + at);
#pragma unroll
            for (int i = 0; i < 4; i++) x[4 * u + i] = z[i];
        }
    };
    auto read_v = [&](int t, int j, float (&x)[8]) RT_INLINE {  // keys 16j + 4hh + 8 (e / 4) + e % 4 of column 32t + col
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int key = 16 * j + 4 * hh + 8 * (e >> 2) + (e & 3);
            x[e] = *(const float*)(Vw + key * ROWB + ((((32 * t + col) >> 2) ^ swizzle(key)) * 16) + 4 * (col & 3));
        }
    };

    float chk = 0.0f;
    uint32_t v_least = ~0u;
    const float* const q_at = Qg + (size_t)min(q_row, Nq - 1) * q_pitch;  // (as in the kernel above)
    Split8 qf[KS];
#pragma unroll
    for (int j = 0; j < KS; j++) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int d = 16 * j + 8 * hh + 4 * u;
            f32x4_t z = *(const f32x4_t*)(q_at + (kExactD ? d : min(d, D - 4)));
            if (!kExactD && d >= D) z = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 4; i++) x[4 * u + i] = z[i];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) chk = split_max(chk, x[i]);
        qf[j] = split8(x);
    }

    f32x16_t acc_o[DT];
    auto zero16 = [](f32x16_t& x) RT_INLINE {
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = 0.0f;
    };
#pragma unroll
    for (int t = 0; t < DT; t++) zero16(acc_o[t]);
    float m_run = neg_inf(), l_run = 0.0f, l_low = 0.0f;

    auto hide = [&](f32x16_t& s, int kv0) RT_INLINE {  // (scaled where the maximum is subtracted)
        if ((kv0 + kTile > N) || (kCausal && kv0 + kTile - 1 > q0)) {
            asm volatile("");  // a branch: the selects cost more than the jump
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int kr = kv0 + 8 * (i >> 2) + 4 * hh + (i & 3);
                if (kr >= N || (kCausal && kr > q_row)) s[i] = neg_inf();
            }
        }
    };
    float alpha = 0.0f;
    auto take_max = [&](const f32x16_t& s) RT_INLINE {
        float m_tile = neg_inf();  // NaN never wins, as in the reference's `if x > m`
#pragma unroll
        for (int i = 0; i < 16; i++) m_tile = __builtin_fmaxf(m_tile, s[i]);
        auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(m_tile), __float_as_uint(m_tile), false, false);
        const float m_new = __builtin_fmaxf(__builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * p.scale, m_run);
        const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
        alpha = (m_run == neg_inf()) ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_use) * kLog2e);
        m_run = m_new;
        return m_use;
    };
    auto add_sum = [&](float tile_l) RT_INLINE {
        const float add = tile_l - l_low * alpha, before = l_run * alpha;
        l_run = before + add;
        l_low = (l_run - before) - add;
    };
    auto rescale = [&]() RT_INLINE {
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc_o[t][i] *= alpha;
        }
    };

    // An operand on its way through the split: eight values, ten steps (two SplitQuads in turn)
    struct Piece {
        float x[8];
        u32x4_t w[3];
        SplitQuad quad;
    };
    auto piece_step = [&](Piece& o, int x, bool is_v) RT_INLINE {
        const int hf = x / SplitQuad::STEPS, k = x % SplitQuad::STEPS;
        if (k == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++) o.quad.r[i] = o.x[4 * hf + i];
        }
        uint32_t a = 0, b2 = 0;
        o.quad.step(k, a, b2);
        if (k % 2 == 0) {
            o.w[k / 2][2 * hf] = a;
            o.w[k / 2][2 * hf + 1] = b2;
        } else if (k == 1) {
            chk = split_max(split_max(chk, o.x[4 * hf]), o.x[4 * hf + 1]);
            chk = split_max(split_max(chk, o.x[4 * hf + 2]), o.x[4 * hf + 3]);
        } else if (is_v) {
#pragma unroll
            for (int i = 0; i < 4; i++) v_least = min(v_least, (__float_as_uint(o.x[4 * hf + i]) << 1) - 1u);
        }
    };
    constexpr int kPiece = 2 * SplitQuad::STEPS;
    constexpr int kPlaneA[6] = {2, 1, 1, 0, 0, 0}, kPlaneC[6] = {0, 1, 0, 2, 1, 0};  // the six terms, the small ones first
    auto frag = [](u32x4_t x) RT_INLINE { return __builtin_bit_cast(bf16x8_t, x); };

    for (int tile = wave; tile < n_tiles; tile += NW) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NREQ) : "memory");  // K; V may still be on its way
        // S, the small terms of all chunks ahead of the large ones; the next chunk of K is split meanwhile
        f32x16_t s;
        zero16(s);
        bf16x8_t head[KS];
        Piece pc[2];
        read_k(0, pc[0].x);
#pragma unroll
        for (int x = 0; x < kPiece; x++) piece_step(pc[0], x, false);
#pragma unroll
        for (int j = 0; j < KS; j++) {
            if (j + 1 < KS) read_k(j + 1, pc[(j + 1) & 1].x);
#pragma unroll
            for (int term = 0; term < 5; term++) {
                s = mfma_h(frag(pc[j & 1].w[kPlaneA[term]]), qf[j].p[kPlaneC[term]], s);
                if (j + 1 < KS) {
#pragma unroll
                    for (int x = term * kPiece / 5; x < (term + 1) * kPiece / 5; x++) piece_step(pc[(j + 1) & 1], x, false);
                }
                RT_ORDER();
            }
            head[j] = frag(pc[j & 1].w[0]);
        }
#pragma unroll
        for (int j = 0; j < KS; j++) s = mfma_h(head[j], qf[j].p[0], s);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // K has been read
        request(k_rsrc, k_lds, tile + NW);
        hide(s, tile * kTile);
        const float m_use = take_max(s);
        rescale();
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NREQ) : "memory");  // V; the next K may be on its way
        read_v(0, 0, pc[0].x);
        u32x4_t pw[2][3];
        float part[2] = {0.0f, 0.0f};
        SplitQuad sp;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            float y[4];
#pragma unroll
            for (int i = 0; i < 4; i++) y[i] = __builtin_fmaf(s[4 * g + i], p.scale, -m_use) * kLog2e;
#pragma unroll
            for (int i = 0; i < 4; i++) sp.r[i] = __builtin_amdgcn_exp2f(y[i]);
#pragma unroll
            for (int i = 0; i < 4; i++) part[i & 1] += sp.r[i];
#pragma unroll
            for (int k = 0; k < SplitQuad::STEPS; k++) {
                uint32_t a = 0, b2 = 0;
                sp.step(k, a, b2);
                if (k % 2) continue;
                pw[g >> 1][k / 2][2 * (g & 1)] = a;
                pw[g >> 1][k / 2][2 * (g & 1) + 1] = b2;
            }
        }
        add_sum(part[0] + part[1]);
#pragma unroll
        for (int x = 0; x < kPiece; x++) piece_step(pc[0], x, true);
        // O: a tile's product in registers of its own, the small terms of both halves of the keys first, then one addition
#pragma unroll
        for (int t = 0; t < DT; t++) {
            f32x16_t o;
            zero16(o);
            read_v(t, 1, pc[1].x);
#pragma unroll
            for (int term = 0; term < 5; term++) {
                o = mfma_h(frag(pc[0].w[kPlaneA[term]]), frag(pw[0][kPlaneC[term]]), o);
#pragma unroll
                for (int x = term * kPiece / 5; x < (term + 1) * kPiece / 5; x++) piece_step(pc[1], x, true);
                RT_ORDER();
            }
            const bf16x8_t head = frag(pc[0].w[0]);
            if (t + 1 < DT) read_v(t + 1, 0, pc[0].x);
#pragma unroll
            for (int term = 0; term < 5; term++) {
                o = mfma_h(frag(pc[1].w[kPlaneA[term]]), frag(pw[1][kPlaneC[term]]), o);
                if (t + 1 < DT) {
#pragma unroll
                    for (int x = term * kPiece / 5; x < (term + 1) * kPiece / 5; x++) piece_step(pc[0], x, true);
                }
                RT_ORDER();
            }
            o = mfma_h(head, frag(pw[0][0]), o);
            o = mfma_h(frag(pc[1].w[0]), frag(pw[1][0]), o);
#pragma unroll
            for (int i = 0; i < 16; i++) acc_o[t][i] += o[i];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // V has been read
        request(v_rsrc, v_lds, tile + NW);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing on its way into LDS that is used otherwise from here on

    bool uncarried = !(chk < kSplitMost);
    if (__any(v_least < kSplitLeast)) {  // small values of V: where a result of this wave's keys is no larger than what they may have lost
        const float least = (l_run + other_half(l_run)) * kSplitLeastResult;
        bool small = false;
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (kExactD || 32 * t + 8 * (i >> 2) + 4 * hh + (i & 3) < D) small |= __builtin_fabsf(acc_o[t][i]) < least;
        uncarried |= small && q_row < Nq && m_run != neg_inf();  // (a row that sees none of them loses nothing)
    }
    if (__syncthreads_or(uncarried)) {
        // something here the split does not carry: the rows once more in f32, out of the same tiles
#pragma unroll
        for (int t = 0; t < DT; t++) zero16(acc_o[t]);
        m_run = neg_inf();
        l_run = l_low = 0.0f;
        float q[16 * DT];
        f32_row<DT>(q, Qg + (size_t)q_row * q_pitch, q_row < Nq, D, hh);
        for (int tile = wave; tile < n_tiles; tile += NW) {
            request(k_rsrc, k_lds, tile);
            request(v_rsrc, v_lds, tile);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            f32x16_t s;
            zero16(s);
#pragma unroll
            for (int j = 0; j < 4 * DT; j++) {  // contraction order 8j + 4hh + i, as f32_row holds the queries
                const f32x4_t a = *(const f32x4_t*)(Kw + col * ROWB + (((2 * j + hh) ^ swizzle(col)) * 16));
#pragma unroll
                for (int i = 0; i < 4; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], q[4 * j + i], s, 0, 0, 0);
            }
            hide(s, tile * kTile);
            const float m_use = take_max(s);
            float tile_l = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], p.scale, -m_use) * kLog2e);
                tile_l += s[i];
            }
            add_sum(tile_l);
            rescale();
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int key = 8 * (i >> 2) + 4 * hh + (i & 3);
#pragma unroll
                for (int t = 0; t < DT; t++) {
                    const float a = *(const float*)(Vw + key * ROWB + ((((32 * t + col) >> 2) ^ swizzle(key)) * 16) + 4 * (col & 3));
                    acc_o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[i], acc_o[t], 0, 0, 0);
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    }

    // ---- the four partial states (as in flash_fwd_f32_splitk_kernel)
    {
        const float l = l_run + other_half(l_run);
        if (hh == 0) {
            red_m[wave][col] = m_run;
            red_l[wave][col] = l;
        }
    }
    __syncthreads();
    float m_all = neg_inf();
#pragma unroll
    for (int w2 = 0; w2 < NW; w2++) m_all = __builtin_fmaxf(m_all, red_m[w2][col]);
    float l_all = 0.0f, my_f = 0.0f;
#pragma unroll
    for (int w2 = 0; w2 < NW; w2++) {
        const float mw = red_m[w2][col];
        const float f = (mw == neg_inf()) ? 0.0f : expf(mw - m_all);  // an empty partial weighs nothing
        l_all += red_l[w2][col] * f;
        if (w2 == wave) my_f = f;
    }
    if (wave == 0 && hh == 0) {
        const bool good = (l_all > 0.0f) && (fabsf(l_all) != __uint_as_float(0x7f800000u)) && (l_all == l_all);
        fin_inv[col] = good ? 1.0f / l_all : quiet_nan();
        if constexpr (DT > 2) {  // (head dims up to 64 keep no statistic here, and a late argument read is 0.3 us of a launch)
            if (p.lse && q_row < Nq) p.lse[((size_t)b * p.heads + h) * (size_t)Nq + q_row] = m_all + logf(l_all);
        }
    }
    float* const Ow = (float*)Kw;  // this wave's weighted O, as rows [col][d]
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            *(f32x4_t*)(Ow + col * LDO + t * 32 + 8 * g + 4 * hh) =
                f32x4_t{acc_o[t][4 * g] * my_f, acc_o[t][4 * g + 1] * my_f, acc_o[t][4 * g + 2] * my_f, acc_o[t][4 * g + 3] * my_f};
    __syncthreads();
#pragma unroll
    for (int n = 0; n < DT; n++) {
        const int idx = 256 * n + tid, r = idx / SL, c = idx % SL;
        f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w2 = 0; w2 < NW; w2++) sum += *(const f32x4_t*)(lds + w2 * 2 * TILE + r * LDO + 4 * c);
        const float inv = fin_inv[r];  // NaN marks a row without a valid sum
        f32x4_t o;
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = (inv == inv) ? sum[i] * inv : quiet_nan();
        if (q0 + r < Nq && 4 * c < D) *(f32x4_t*)(Og + (size_t)(q0 + r) * o_pitch + 4 * c) = o;
    }
}

}  // namespace

hipError_t launch_flash_f32_split(hipStream_t stream, const FlashF32Params& p_in) {
    FlashF32Params p = p_in;
    dim3 grid((p.seq + 4 * kTile - 1) / (4 * kTile), p.heads, p.batch), block(256);
    // Causal rows are of unequal length.  Up to head dim 64 two workgroups share a CU: where all are resident at once the
    // pairs are made by place.  Above, one fills a CU (LDS), and left to the order of the launch the long blocks of a later
    // head met the long ones before them: two blocks a workgroup (B=4 H=16 N=1024 D=128 203 -> 133 us).
    const long long n = (long long)grid.x * grid.y * grid.z;
    p.zigzag = 0;
    if (p.mask == kMaskCausal && p.dim <= 64 && n <= 2ll * p.n_cus) p.zigzag = 1;
    if (p.mask == kMaskCausal && p.dim > 64 && n > p.n_cus) {
        p.zigzag = 2;
        grid.x = (grid.x + 1) / 2;
    }
    deal_to_xcds(p, grid.x);
    auto launch = [&](auto dt_c, auto exact_c) {
        constexpr int kDT = decltype(dt_c)::value;
        constexpr bool kEx = decltype(exact_c)::value;
        if (p.mask == kMaskCausal) hipLaunchKernelGGL((flash_fwd_f32_split_kernel<kDT, kEx, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((flash_fwd_f32_split_kernel<kDT, kEx, false>), grid, block, 0, stream, p);
    };
    auto launch_dt = [&](auto dt_c) {
        if (p.dim % 32 == 0) launch(dt_c, std::true_type{});
        else launch(dt_c, std::false_type{});
    };
    switch ((p.dim + 31) / 32) {
        case 1: launch_dt(std::integral_constant<int, 1>{}); break;
        case 2: launch_dt(std::integral_constant<int, 2>{}); break;
        case 3: launch_dt(std::integral_constant<int, 3>{}); break;
        case 4: launch_dt(std::integral_constant<int, 4>{}); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

bool flash_f32_split_keys_supported(const FlashF32Params& p) {
    const long long keys = p.seq_kv ? p.seq_kv : p.seq;
    return p.dim <= 128 && p.dim % 4 == 0 && (p.mask == kMaskNone || p.mask == kMaskCausal) && !p.bias && (!p.lse || p.dim > 64) && keys > 0 &&
           (unsigned long long)(keys + 256) * (unsigned long long)p.lkv.row_pitch * 4ull < (1ull << 32);  // 32-bit offsets
}

hipError_t launch_flash_f32_split_keys(hipStream_t stream, const FlashF32Params& p_in) {
    FlashF32Params p = p_in;
    if (!flash_f32_split_keys_supported(p)) return hipErrorInvalidValue;
    dim3 grid((p.seq + kTile - 1) / kTile, p.heads, p.batch), block(256);
    p.zigzag = (p.mask == kMaskCausal) && ((long long)grid.x * grid.y * grid.z <= (p.dim <= 64 ? 2ll : 1ll) * p.n_cus) ? 1 : 0;
    deal_to_xcds(p, grid.x);
    auto launch = [&](auto dt_c, auto exact_c) {
        constexpr int kDT = decltype(dt_c)::value;
        constexpr bool kEx = decltype(exact_c)::value;
        if (p.mask == kMaskCausal) hipLaunchKernelGGL((flash_fwd_f32_split_keys_kernel<kDT, kEx, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((flash_fwd_f32_split_keys_kernel<kDT, kEx, false>), grid, block, 0, stream, p);
    };
    auto launch_dt = [&](auto dt_c) {
        if (p.dim % 32 == 0) launch(dt_c, std::true_type{});
        else launch(dt_c, std::false_type{});
    };
    switch ((p.dim + 31) / 32) {
        case 1: launch_dt(std::integral_constant<int, 1>{}); break;
        case 2: launch_dt(std::integral_constant<int, 2>{}); break;
        case 3: launch_dt(std::integral_constant<int, 3>{}); break;
        case 4: launch_dt(std::integral_constant<int, 4>{}); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace rt
