// f32 flash-attention forward for gfx950: the device counterpart of
// flash_forward_masked (crates/rustorch-attention/src/cpu_forward.rs:193-425) and of the
// prefill branch of gqa_forward_f32 (crates/rustorch-nn/src/gqa.rs:151-177).
//
// One wavefront owns 32 query rows and walks the key/value rows 32 at a time.  Both
// products run on the f32 matrix cores (v_mfma_f32_32x32x2_f32, full f32 precision):
//
//   S^T[kv, q]  = sum_d K[kv, d] * Q[q, d]          (A = K tile, B = Q tile)
//   O^T[d, q]  += sum_kv V[kv, d] * P[q, kv]        (A = V tile, B = P from registers)
//
// Computing the transposed score tile leaves every lane holding 16 scores of ONE query row
// (q = lane % 32), so the row max / row sum of the online softmax are in-lane reductions plus
// one exchange with the other half of the wave, and the score registers are already in the
// B-operand layout the second product needs: P never leaves the register file.
//
// Semantics kept from the reference: scale applied to the finished dot product, mask -> -inf
// after scaling, row without a visible key -> NaN row, `out = O * (1/l)`.  Tiles a causal mask
// empties are skipped, not computed.
#include <type_traits>

#include "rt_common.hpp"
#include "rt_kernels.hpp"

namespace rt {

namespace {

constexpr int kRows = 32;  // query rows per workgroup (one wave) and key rows per step

template <int DT>  // DT = ceil(dim / 32); the head dim is zero-padded to DPAD = 32 * DT in LDS
__global__ __launch_bounds__(64) void flash_fwd_f32_kernel(FlashF32Params p) {
    constexpr int DPAD = 32 * DT;
    constexpr int LDQ = DPAD + 1;  // odd row stride: a column read (32 rows, fixed d) hits 32 banks
    __shared__ float Qs[kRows * LDQ];
    __shared__ float Ks[kRows * LDQ];
    __shared__ float Vs[kRows * DPAD];  // read along d: no padding needed

    const int lane = threadIdx.x;
    const int col = lane & 31;  // query row within the tile / MFMA column
    const int hh = lane >> 5;   // which half of the wave
    const int N = p.seq, D = p.dim;
    const int qtile = (int)gridDim.x - 1 - (int)blockIdx.x;  // longest causal rows first
    const int q0 = qtile * kRows;
    const int h = blockIdx.y, b = blockIdx.z;
    const int kvh = h / p.group;
    const float* __restrict__ Qg = p.q + (size_t)b * p.lq.batch_stride + (size_t)h * p.lq.head_stride;
    const float* __restrict__ Kg = p.k + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    const float* __restrict__ Vg = p.v + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    float* __restrict__ Og = p.out + (size_t)b * p.lo.batch_stride + (size_t)h * p.lo.head_stride;
    const size_t q_pitch = p.lq.row_pitch, kv_pitch = p.lkv.row_pitch, o_pitch = p.lo.row_pitch;

    // With a padding mask the reference's recurrence turns every row into NaN when its first
    // key tile [0, bc) holds no visible key (cpu_forward.rs:364-384); reproduce that outcome.
    bool poison = false;
    if (p.mask == kMaskPadding) {
        int lim = p.ref_bc < N ? p.ref_bc : N;
        bool any = false;
        for (int j = lane; j < lim; j += kWave) any |= (p.keep[j] != 0);
        poison = !__any(any);
    }

    // stage the Q tile (zero beyond seq and beyond dim)
    for (int idx = lane; idx < kRows * DPAD; idx += kWave) {
        int r = idx / DPAD, d = idx - r * DPAD;
        int qr = q0 + r;
        Qs[r * LDQ + d] = (qr < N && d < D) ? Qg[(size_t)qr * q_pitch + d] : 0.0f;
    }

    f32x16_t acc_o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc_o[t][i] = 0.0f;
    float m_run = neg_inf();
    float l_run = 0.0f;  // this lane's share of the row sum (its 16 keys per step)

    const int q_row = q0 + col;
    int kv_end = N;
    if (p.mask == kMaskCausal) kv_end = min(N, q0 + kRows);  // keys beyond the tile's last row are masked

    for (int kv0 = 0; kv0 < kv_end; kv0 += kRows) {
        __syncthreads();
        for (int idx = lane; idx < kRows * DPAD; idx += kWave) {
            int r = idx / DPAD, d = idx - r * DPAD;
            int kr = kv0 + r;
            bool ok = (kr < N && d < D);
            Ks[r * LDQ + d] = ok ? Kg[(size_t)kr * kv_pitch + d] : 0.0f;
            Vs[r * DPAD + d] = ok ? Vg[(size_t)kr * kv_pitch + d] : 0.0f;
        }
        __syncthreads();

        // S^T = K . Q^T
        f32x16_t s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.0f;
#pragma unroll 8
        for (int ks = 0; ks < DPAD / 2; ks++) {
            float a = Ks[col * LDQ + 2 * ks + hh];
            float bq = Qs[col * LDQ + 2 * ks + hh];
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(a, bq, s, 0, 0, 0);
        }
        // register i of the accumulator holds key row 8*(i/4) + 4*hh + (i%4), query row `col`
        float m_tile = neg_inf();
#pragma unroll
        for (int i = 0; i < 16; i++) {
            int kr = kv0 + 8 * (i >> 2) + 4 * hh + (i & 3);
            float x = s[i] * p.scale;
            bool masked = kr >= N;
            if (p.mask == kMaskCausal) masked |= kr > q_row;
            if (p.mask == kMaskPadding) masked |= (kr < N) && (p.keep[kr] == 0);
            x = masked ? neg_inf() : x;
            s[i] = x;
            m_tile = (x > m_tile) ? x : m_tile;  // NaN never wins, as in the reference's `if x > m`
        }
        {
            float o = other_half(m_tile);
            m_tile = (o > m_tile) ? o : m_tile;
        }
        float m_new = (m_tile > m_run) ? m_tile : m_run;
        // No branch here: MFMA ignores the exec mask, so every lane must reach the products with
        // well-defined operands.  While a row has seen no visible key, subtract 0 instead of -inf:
        // every exp() is then exp(-inf) = 0 and the state stays empty.
        float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
        float alpha = (m_run == neg_inf()) ? 0.0f : expf(m_run - m_use);
        m_run = m_new;
        float tile_l = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float e = expf(s[i] - m_use);
            s[i] = e;
            tile_l += e;
        }
        l_run = l_run * alpha + tile_l;
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc_o[t][i] *= alpha;

        // O^T += V^T . P^T, two keys per MFMA: the lower half of the wave feeds key 8j+r, the upper 8j+4+r
#pragma unroll
        for (int i = 0; i < 16; i++) {
            int kr = 8 * (i >> 2) + 4 * hh + (i & 3);
#pragma unroll
            for (int t = 0; t < DT; t++) {
                float a = Vs[kr * DPAD + t * 32 + col];
                acc_o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[i], acc_o[t], 0, 0, 0);
            }
        }
    }

    float l = l_run + other_half(l_run);
    bool good = (l > 0.0f) && (fabsf(l) != __uint_as_float(0x7f800000u)) && (l == l) && !poison;
    float inv_l = 1.0f / l;
    if (p.lse && hh == 0 && q_row < N) p.lse[((size_t)b * p.heads + h) * (size_t)N + q_row] = m_run + logf(l);
    if (q_row < N) {
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                int d = t * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
                if (d < D) Og[(size_t)q_row * o_pitch + d] = good ? acc_o[t][i] * inv_l : quiet_nan();
            }
    }
}


// ---- head dims that are a multiple of 32, 16-byte aligned rows: the fast kernel ---------------------------
//
// One workgroup of four waves owns 32 query rows; wave w walks the key tiles t = w, w+4, ... (32 keys each) on its
// own, with a private LDS tile and no workgroup barrier in the loop, and the four partial (O, m, l) states are
// merged through LDS at the end with the online-softmax monoid (online_softmax.rs:105-131 extended with O).
// Splitting the keys rather than the query rows over the waves shortens the longest chain of dependent steps
// four times, which is what a small problem (8 heads x 2048 rows) is bound by.  The next tile travels from
// global memory into registers (16-byte loads) while the current one is multiplied.
//
// The contraction index of the score product is walked in the order d = 8j + 4*half + i (i = 0..3) for both
// operands, so that a lane fetches its four K values of a chunk with one 16-byte LDS read and Q stays in
// registers for the whole job.
// kExactD: dim == 32 * DT, no column guards anywhere.  kMode: one instantiation per way of masking, so that the tile
// step of each holds only its own tests -- 0 none, 1 causal, 2 Mask::Padding (the only one that carries the keep
// bits in LDS and looks at p.keep), 3 none plus an additive score bias.
template <int DT, bool kExactD, int kMode>
__global__ __launch_bounds__(256, (DT <= 2 ? 2 : 1)) void flash_fwd_f32_splitk_kernel(FlashF32Params p) {
    constexpr bool kCausal = kMode == 1, kPad = kMode == 2, kBias = kMode == 3;
    constexpr int DPAD = 32 * DT;       // dim rounded up to a multiple of 32 (columns beyond dim are zeros in LDS)
    constexpr int LDK = DPAD + 4;       // row stride of the K tile: 16-byte reads of 16 rows tile all banks
    constexpr int CH = DPAD / 4;        // 16-byte chunks per row
    constexpr int NLD = 32 * CH / 64;   // 16-byte loads per lane, per matrix, per tile
    constexpr int KTILE = kRows * LDK, VTILE = kRows * DPAD;
    constexpr int NW = 4;
    __shared__ __attribute__((aligned(16))) float lds[NW * (KTILE + VTILE)];
    __shared__ float red_m[NW][kRows], red_l[NW][kRows];
    __shared__ float fin_inv[kRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    // the arguments, requested together: left to itself the compiler loads a field where it is first used, and waits for it there
    asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.out), "s"(p.lse), "s"(p.heads), "s"(p.group), "s"(p.seq), "s"(p.seq_kv), "s"(p.dim), "s"(p.scale),
                 "s"(p.zigzag), "s"(p.dealt), "s"(p.blocks_magic), "s"(p.heads_magic), "s"(p.lq.batch_stride), "s"(p.lq.head_stride), "s"(p.lq.row_pitch));
    asm volatile("" ::"s"(p.lkv.batch_stride), "s"(p.lkv.head_stride), "s"(p.lkv.row_pitch), "s"(p.lo.batch_stride), "s"(p.lo.head_stride), "s"(p.lo.row_pitch));
    const int Nq = p.seq, N = p.seq_kv ? p.seq_kv : p.seq;  // N: keys (== queries unless cross-attention)
    const int D = kExactD ? DPAD : p.dim;
    // Which (batch, head, query tile) this workgroup takes.  Workgroups are dealt round-robin to the 8 XCDs, each
    // with its own L2: when the heads divide evenly, XCD x takes the heads bh = x (mod 8) and walks them one after
    // the other, longest causal rows first, so that a head's K and V are fetched into one L2 only.  When the whole
    // grid is resident at once (p.zigzag) the second half of an XCD's list runs shortest-first, so that the two
    // workgroups that end up sharing a CU (list positions r and r + half) are a long one and a short one.
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
    const int q0 = qtile * kRows;
    const int kvh = p.group == 1 ? h : h / p.group;
    const float* __restrict__ Qg = p.q + (size_t)b * p.lq.batch_stride + (size_t)h * p.lq.head_stride;
    const float* __restrict__ Kg = p.k + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    const float* __restrict__ Vg = p.v + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    float* __restrict__ Og = p.out + (size_t)b * p.lo.batch_stride + (size_t)h * p.lo.head_stride;
    const size_t q_pitch = p.lq.row_pitch, kv_pitch = p.lkv.row_pitch, o_pitch = p.lo.row_pitch;
    float* Kw = lds + wave * (KTILE + VTILE);
    float* Vw = Kw + KTILE;

    // leading-masked-tile rule of the reference's recurrence (cpu_forward.rs:364-384), as in the kernel above
    bool poison = false;
    // The keep vector as one bit per key in LDS (up to 32 * kKeepWords keys; longer ones are read byte by byte in the
    // loop): a tile step then reads one word, and a tile without a hidden key is not masked at all.
    constexpr int kKeepWords = 1024;
    __shared__ uint32_t keep_bits[kPad ? kKeepWords : 2];
    const bool keep_in_lds = kPad && N <= 32 * kKeepWords;
    if constexpr (kPad) {
        int lim = p.ref_bc < N ? p.ref_bc : N;
        bool any = false;
        for (int j = lane; j < lim; j += kWave) any |= (p.keep[j] != 0);
        poison = !__any(any);
        if (keep_in_lds) {
            for (int base = wave * kWave; base < N; base += NW * kWave) {
                const int key = base + lane;
                const unsigned long long bal = __ballot(key < N && p.keep[key] != 0);
                if (lane == 0) {
                    keep_bits[base >> 5] = (uint32_t)bal;
                    keep_bits[(base >> 5) + 1] = (uint32_t)(bal >> 32);
                }
            }
            __syncthreads();
        }
    }

    const int q_row = q0 + col;
    f32x16_t acc_o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc_o[t][i] = 0.0f;
    float m_run = neg_inf();
    float l_run = 0.0f;  // this lane's share of the row sum

    int kv_end = N;
    if (kCausal) kv_end = min(N, q0 + kRows);
    const int n_tiles = (kv_end + kRows - 1) / kRows;
    // additive bias row of this lane's query (MultiHeadAttention's attn_mask, added to the scaled scores)
    const float* __restrict__ bias_row = nullptr;
    if (kBias && q_row < Nq)
        bias_row = p.bias + ((size_t)b * p.heads + h) * (size_t)p.bias_bh_stride + (size_t)q_row * (size_t)N;
    const bool bias_vec = ((N & 3) == 0) && ((((uintptr_t)p.bias) & 15) == 0) && ((p.bias_bh_stride & 3) == 0);

    // lane's chunks of a tile: load n covers row (64n + lane) / CH, chunk (64n + lane) % CH.  When CH divides 64
    // that is row n * (64/CH) + lane / CH, chunk lane % CH: one per-lane offset, everything else is uniform.
    constexpr bool kEvenRows = (64 % CH == 0);
    constexpr int RPL = kEvenRows ? 64 / CH : 0;  // rows per load instruction
    const int ld_r = lane / CH, ld_c = lane % CH;
    const bool ld_col_ok = kExactD || 4 * ld_c < D;  // this lane's 16-byte column exists
    const uint32_t ld_off = (uint32_t)ld_r * (uint32_t)kv_pitch * 4u + (uint32_t)ld_c * 16u;  // bytes; a few rows: fits
    // Through descriptors that end with the tile's last key: a row behind it and a column behind the head dim come back as zeros
    // without a read, and no load stands behind a test of its own.  The wave's number is known to be uniform: where it was not, each
    // request was a loop over the lanes that agree on a descriptor.  us, so (whole tiles through pointers) -> now, B H N head dim: causal 1 4 30 128 10.4 ->
    // 8.8, 1 8 40 32 5.5 -> 5.1; unmasked 1 8 161 128 16.8 -> 15.8, 1 8 250 20 7.4 -> 6.8, 1 8 60 96 9.0 -> 8.1, with the row statistic 3 5 777 32 24.5
    // -> 23.4; a padding mask 1 8 2048 64 89.7 -> 82.1, 2 8 777 64 41.5 -> 37.3, 2 8 600 96 60.1 -> 54.2.
    f32x4_t kreg[NLD], vreg[NLD];
    const uint32_t pitch_b = (uint32_t)kv_pitch * 4u;
    auto issue_loads = [&](int tile) {
        const size_t base = (size_t)tile * kRows * kv_pitch;
        const uint32_t bytes = (uint32_t)(min(N - tile * kRows, kRows) - 1) * pitch_b + 4u * (uint32_t)D;
        const __amdgpu_buffer_rsrc_t kb = __builtin_amdgcn_make_buffer_rsrc((void*)(Kg + base), 0, bytes, kBufferFlags);
        const __amdgpu_buffer_rsrc_t vb = __builtin_amdgcn_make_buffer_rsrc((void*)(Vg + base), 0, bytes, kBufferFlags);
#pragma unroll
        for (int n = 0; n < NLD; n++) {
            uint32_t off, step = 0;
            if constexpr (kEvenRows) {
                off = ld_col_ok ? ld_off : 0x7fffffffu;
                step = (uint32_t)(RPL * n) * pitch_b;  // uniform
            } else {
                const int idx = 64 * n + lane, r = idx / CH, c = idx % CH;
                off = kExactD || 4 * c < D ? (uint32_t)r * pitch_b + 16u * (uint32_t)c : 0x7fffffffu;
            }
            kreg[n] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(kb, off, step, 0));
            vreg[n] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(vb, off, step, 0));
        }
    };
    if (wave < n_tiles) issue_loads(wave);

    // Q as B operand, in registers (requested behind the first tile): qreg[4j + i] = Q[q0 + col][8j + 4hh + i]
    const float* const q_at = Qg + (size_t)min(q_row, Nq - 1) * q_pitch;  // (a row behind the last repeats it and is not written)
    float qreg[DPAD / 2];
#pragma unroll
    for (int j = 0; j < DPAD / 8; j++) {
        const int d = 8 * j + 4 * hh;
        f32x4_t z = *(const f32x4_t*)(q_at + (kExactD ? d : min(d, D - 4)));
        if (!kExactD && d >= D) z = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; i++) qreg[4 * j + i] = z[i];
    }

    for (int tile = wave; tile < n_tiles; tile += NW) {
        const int kv0 = tile * kRows;
        // registers -> this wave's LDS tile (its reads of the previous tile are behind it: same wave, in order)
#pragma unroll
        for (int n = 0; n < NLD; n++) {
            const int idx = 64 * n + lane, r = idx / CH, c = idx % CH;
            *(f32x4_t*)(Kw + r * LDK + 4 * c) = kreg[n];
            *(f32x4_t*)(Vw + r * DPAD + 4 * c) = vreg[n];
        }
        // this tile's bias values are requested ahead of the next tile's rows: a wait for them then leaves the
        // prefetch in flight (requests complete in order)
        f32x16_t bias;
#pragma unroll
        for (int i = 0; i < 16; i++) bias[i] = 0.0f;
        if (kBias && bias_row) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int kr0 = kv0 + 8 * g + 4 * hh;
                if (bias_vec && kr0 + 3 < N) {
                    const f32x4_t bv = *(const f32x4_t*)(bias_row + kr0);
#pragma unroll
                    for (int r = 0; r < 4; r++) bias[4 * g + r] = bv[r];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (kr0 + r < N) bias[4 * g + r] = bias_row[kr0 + r];
                }
            }
        }
        if (tile + NW < n_tiles) issue_loads(tile + NW);

        // S^T = K . Q^T
        f32x16_t s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < DPAD / 8; j++) {
            const f32x4_t a = *(const f32x4_t*)(Kw + col * LDK + 8 * j + 4 * hh);
#pragma unroll
            for (int i = 0; i < 4; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], qreg[4 * j + i], s, 0, 0, 0);
        }
        // register i of the accumulator holds key row 8*(i/4) + 4*hh + (i%4), query row `col`
        float m_tile = neg_inf();
        const uint32_t keep_word = keep_in_lds ? keep_bits[kv0 >> 5] : 0u;  // bit r: key kv0 + r is visible
        const bool edge = (kv0 + kRows > N) || (kCausal && kv0 + kRows - 1 > q0) ||
                          (kPad && keep_word != 0xffffffffu);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float x = kBias ? s[i] * p.scale + bias[i] : s[i] * p.scale;
            if (edge) {
                int kr = kv0 + 8 * (i >> 2) + 4 * hh + (i & 3);
                bool masked = kr >= N;
                if (kCausal) masked |= kr > q_row;
                if constexpr (kPad) {
                    if (keep_in_lds) masked |= ((keep_word >> (8 * (i >> 2) + 4 * hh + (i & 3))) & 1u) == 0;
                    else masked |= (kr < N) && (p.keep[kr] == 0);
                }
                x = masked ? neg_inf() : x;
            }
            s[i] = x;
            m_tile = (x > m_tile) ? x : m_tile;  // NaN never wins, as in the reference's `if x > m`
        }
        {
            // the two halves of the wave hold the same query rows: v_permlane32_swap leaves the lower halves' values
            // in one register and the upper halves' in the other, without a trip through LDS (neither is NaN)
            auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(m_tile), __float_as_uint(m_tile), false, false);
            const float lo = __uint_as_float(r[0]), hi = __uint_as_float(r[1]);
            m_tile = (hi > lo) ? hi : lo;
        }
        float m_new = (m_tile > m_run) ? m_tile : m_run;
        float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
        float alpha = (m_run == neg_inf()) ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_use) * kLog2e);
        m_run = m_new;
        // exp(x) as exp2(x * log2 e) on the hardware exp2: the difference is taken first (exact for the terms
        // that matter), so the argument carries one rounding, about 1e-7 relative on each weight
        float part[4];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float e = __builtin_amdgcn_exp2f((s[i] - m_use) * kLog2e);
            s[i] = e;
            if (i < 4) part[i] = e;
            else part[i & 3] += e;
        }
        l_run = l_run * alpha + ((part[0] + part[1]) + (part[2] + part[3]));
        if (__any(alpha != 1.0f)) {  // wave-uniform: the reference also rescales only when alpha != 1 (cpu_forward.rs:372)
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc_o[t][i] *= alpha;
        }
        // O^T += V^T . P^T, two keys per instruction: the lower half of the wave feeds key 8j+r, the upper 8j+4+r
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int kr = 8 * (i >> 2) + 4 * hh + (i & 3);
#pragma unroll
            for (int t = 0; t < DT; t++) {
                float a = Vw[kr * DPAD + t * 32 + col];
                acc_o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[i], acc_o[t], 0, 0, 0);
            }
        }
    }

    // ---- merge the four partial states
    {
        float l = l_run + other_half(l_run);
        if (hh == 0) {
            red_m[wave][col] = m_run;
            red_l[wave][col] = l;
        }
    }
    __syncthreads();  // also: every wave is done with its tiles
    float m_all = neg_inf();
#pragma unroll
    for (int w2 = 0; w2 < NW; w2++) {
        float mw = red_m[w2][col];
        m_all = (mw > m_all) ? mw : m_all;
    }
    float l_all = 0.0f, my_f = 0.0f;
#pragma unroll
    for (int w2 = 0; w2 < NW; w2++) {
        float mw = red_m[w2][col];
        float f = (mw == neg_inf()) ? 0.0f : expf(mw - m_all);  // an empty partial weighs nothing
        l_all += red_l[w2][col] * f;
        if (w2 == wave) my_f = f;
    }
    if (wave == 0 && hh == 0) {
        bool good = (l_all > 0.0f) && (fabsf(l_all) != __uint_as_float(0x7f800000u)) && (l_all == l_all) && !poison;
        fin_inv[col] = good ? 1.0f / l_all : quiet_nan();
        if (p.lse && q0 + col < Nq) p.lse[((size_t)b * p.heads + h) * (size_t)Nq + q0 + col] = m_all + logf(l_all);
    }
    // this wave's weighted O, as rows [col][d], into its own K tile
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4_t o = {acc_o[t][4 * g] * my_f, acc_o[t][4 * g + 1] * my_f, acc_o[t][4 * g + 2] * my_f, acc_o[t][4 * g + 3] * my_f};
            *(f32x4_t*)(Kw + col * LDK + t * 32 + 8 * g + 4 * hh) = o;
        }
    __syncthreads();
    // all 256 threads: sum the four partial tiles, normalise, store whole rows
#pragma unroll
    for (int n = 0; n < (kRows * CH + 255) / 256; n++) {
        const int idx = 256 * n + tid;
        if (idx < kRows * CH) {
            const int r = idx / CH, c = idx % CH;
            f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w2 = 0; w2 < NW; w2++) sum += *(const f32x4_t*)(lds + w2 * (KTILE + VTILE) + r * LDK + 4 * c);
            const float inv = fin_inv[r];
            // a NaN in fin_inv marks a row without a valid sum: the whole row is NaN, whatever O holds
            f32x4_t o;
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = (inv == inv) ? sum[i] * inv : quiet_nan();
            if (q0 + r < Nq && 4 * c < D) *(f32x4_t*)(Og + (size_t)(q0 + r) * o_pitch + 4 * c) = o;
        }
    }
}

}  // namespace

// Which of the two kernels has less to do on its busiest SIMD, in tile steps of this file's kernel.  The split kernel owns 128
// rows a workgroup and walks all their keys.
//
// Causal, and head dims above 64: this file's kernel spreads 32-row workgroups whose waves share the keys, so it is near the
// mean of the chip; the split kernel takes 0.58 of the time per step at head dim 64 (1.6 against 2.83 us per tile of 32 x 32
// and SIMD) and 0.68 at 32 (1.08 against 1.6); half a step more of fixed cost here.  us here / there, head dim 64 causal: one
// sequence of 8 heads, 2048 keys 52 / 91, 4096 159 / 173; 2 x 12 heads, 999 keys 46 / 49; 8 x 16 heads, 256 keys 27 / 19.
// Head dim 128: 8 heads, 2048 keys 178 / 174, 16 heads, 1500 keys 203 / 122; 4 x 16 heads, 1024 keys 395 / 198, causal
// 239 / 119.
//
// Without a mask up to head dim 64 the gradients follow the same rule, so that they form the scores in the order in which the
// row statistic was formed, and the line lies where forward and gradients together break even.  Every workgroup has the
// same to do there: rounds of 32-row workgroups (one a CU in the gradients at head dim 64, two at 32) with a quarter of the
// tiles each, against rounds of 128-row ones at 0.5 (0.345) of a step.  us here / there, forward and gradients (in a launch each), B H N
// at head dim 64: 4 12 283 72 / 70, 8 16 200 107 / 64, 1 12 1500 395 / 256; at 32: 4 12 300 46 / 55, 8 16 200 59 / 40, 4 16 1024 336 / 234;
// with the gradients in one launch (flash_f32_gradients_join) 4 8 256 34 / 47, 4 8 128 18 / 28.
static bool flash_f32_split_pays(const FlashF32Params& p) {
    const double n_cus = p.n_cus > 0 ? p.n_cus : 256;
    const long long keys = p.seq_kv ? p.seq_kv : p.seq;
    const double tiles = (double)((keys + 31) / 32), blocks = (p.seq + 127) / 128, n_bh = (double)p.heads * p.batch;
    const bool causal = p.mask == kMaskCausal;
    const double per_cu = n_bh * blocks / n_cus;
    if (!causal && p.dim <= 64) {
        const double rounds = __builtin_ceil(n_bh * ((p.seq + 31) / 32) / (p.dim > 32 ? n_cus : 2 * n_cus));
        return __builtin_ceil(per_cu) * tiles * (p.dim > 32 ? 0.5 : 0.345) < 1.02 * rounds * __builtin_ceil(tiles / 4) - 0.2;
    }
    const double here = n_bh * ((p.seq + 31) / 32) * (causal ? (tiles + 1) / 2 : tiles) / (4 * n_cus);
    double there = __builtin_ceil(per_cu) * tiles;
    if (causal) {
        if (p.dim <= 64) there = __builtin_fmax(tiles, 1.1 * per_cu * (tiles + 4) / 2);
        else there = per_cu > 1 ? __builtin_ceil(per_cu / 2) * (tiles + 4) : tiles;  // two blocks a workgroup
    }
    return there * (p.dim > 64 ? 0.55 : (p.dim > 32 ? 0.58 : 0.68)) < here + 0.5;
}

// The same question between the two forms of the split products (flash_f32_split.hip: 128 query rows a workgroup, or 32 and
// waves that share the keys), for a forward without row statistic, in us beside the launch.  At head
// dim 64 a tile step of 128 rows takes 1.41 us (1.45 causal, with what its rows of unequal length leave idle), one of the
// four waves' 3.8 with two workgroups on a CU and 2.2 with one; causal 1.9 a step of the chip's mean and 2.3 for each
// workgroup of a CU; at 32 0.87 and 1.05, causal 1.02 and 1.05 with 1.3 a workgroup.  us, 128 rows / shared keys, B H N at
// head dim 64: 1 8 2048 94 / 69, causal 91 / 43; 8 8 256 17.0 / 14.5; 2 12 400 23 / 19; 1 12 1500 69 / 72; 5 12 300 20 / 25; 4 16 1024
// 95 / 129, causal 63 / 85; causal 1 8 4096 173 / 128, 2 12 999 49 / 38, 4 16 512 29 / 32, 8 16 256 19 / 24; at 32: 8 16 300 24 / 21,
// 4 16 1024 63 / 73, causal 1 8 4096 144 / 78, 2 16 2048 80 / 83.
// Above head dim 64 one workgroup of either form fills a CU.  Causal, a tile step of 128 rows takes 2.45 us (2.8 above 96), one of the
// four waves' 3.6 (4.5), and a workgroup of them 4.5 (5.5) beside its steps; blocks of 128 rows go two to a workgroup
// from one a CU on, those of 32 come near the chip's mean but for the longest.  Unmasked 2.45 (2.65) and 6.2 (6.5) a launch, against 2.85 (3.9), 5.6
// a workgroup (6.8, and 8 between 96 and 128) and 1.2 (0.5): fitted to 110 drawn calls near the line and held against 70 others, of which the
// slower form is taken by 2 to 5 % in three.  us, f32 kernel / 128 rows / shared keys, B H N at head dim 128: 1 8 2048 178 / 174 / 145; 2 8 1024
// 95 / 92 / 81; 4 8 400 52 / 44 / 48; 2 12 700 107 / 67 / 94; 1 8 161 15.7 / 24.6 / 15.6; 128 rows / shared keys 3 16 248 28.2 / 30.1, 1 16 575 51.0 / 52.0, 1 32/8
// 371 37.7 / 37.6, 1 12 1185 100 / 91; at 100 2 12 337 34.3 / 38.9, 1 8 1751 140 / 125; at 80 2 32/8 206 23.2 / 24.2, 2 16 308 30.1 / 29.4; at 68 3 8 1556
// 238 / 213.  Causal 1 8 3438 271 / 284 / 223; 1 12 1500 133 / 128 / 109; 1 16 2048 196 / 175 / 168; 2 16 1500 236 / 156 / 206; unmasked at 96 1 8 1024 39.7 / 82.7 /
// 29.9; 8 8 200 26.3 / 25.8 / 25.7; 1 16 2048 288 / 163 / 216; causal 2 12 999 84 / 85 / 70; 4 12 600 67 / 55 / 61.
static bool flash_f32_rows_pay(const FlashF32Params& p) {
    const double n_cus = p.n_cus > 0 ? p.n_cus : 256;
    const long long keys = p.seq_kv ? p.seq_kv : p.seq;
    const double tiles = (double)((keys + 31) / 32), n_bh = (double)p.heads * p.batch, groups = n_bh * ((p.seq + 31) / 32);
    const double per_cu = n_bh * ((p.seq + 127) / 128) / n_cus, share = __builtin_ceil(tiles / 4);
    if (p.dim > 64) {
        const bool high = p.dim > 96;
        if (p.mask == kMaskCausal) {
            const double row_step = high ? 2.8 : 2.45, key_step = high ? 4.5 : 3.6, own = high ? 5.5 : 4.5;
            return row_step * (per_cu > 1 ? __builtin_ceil(per_cu / 2) * (tiles + 4) : tiles) <
                   __builtin_fmax(key_step * share, key_step * groups * (tiles + 1) / (8 * n_cus) + own * groups / n_cus);
        }
        const double each = high ? (p.dim == 128 ? 6.8 : 8.0) : 5.6;
        return (high ? 2.65 : 2.45) * __builtin_ceil(per_cu) * tiles + (high ? 6.5 : 6.2) <
               __builtin_ceil(groups / n_cus) * ((high ? 3.9 : 2.85) * share + each) + (high ? 0.5 : 1.2);
    }
    if (p.mask == kMaskCausal) {
        const double rows = __builtin_fmax(tiles, 1.1 * per_cu * (tiles + 4) / 2), mean = groups * (tiles + 1) / (8 * n_cus);
        return p.dim > 32 ? 1.45 * rows < 1.9 * mean + 2.3 * groups / n_cus : 1.02 * rows + 2 < 1.05 * mean + 1.3 * groups / n_cus;
    }
    const double rows = __builtin_ceil(per_cu) * tiles;
    if (p.dim <= 32) return 0.87 * rows < 1.05 * share * groups / n_cus;
    const double full = __builtin_floor(groups / (2 * n_cus)), rest = groups - full * 2 * n_cus;
    return 1.41 * rows < share * (3.8 * full + (rest > n_cus ? 3.8 : (rest > 0 ? 2.2 : 0.0)));
}

// Keys from which the shared keys pay: with 128 a wave has one tile at most, and the f32 kernel is ahead (1 8 128 at head dim 64 6.6 / 7.3 us, 96
// 8.9 / 9.3, 128 10.2 / 11.6, and with two tiles a wave at most nearly level there: 1 8 160 15.6 / 15.5, 224 16.2 / 15.6; at 64 1 8 161 9.5 / 9.3).
// Unmasked up to head dim 32 it is level up to 256 (us, f32 kernel / shared keys, B H N: 1 8 256 6.9 / 6.8, 2 12 256 7.0 / 6.9,
// 8 8 256 10.0 / 9.4) and keeps those calls, which then give the bits of the forward that keeps its row statistic; against
// 128 rows a workgroup they pay there as well (1 8 160 10.5 / 6.7).
constexpr int kSplitKeysFrom = 129, kSplitKeysFrom32 = 257, kSplitKeysFrom128 = 225;
static bool flash_f32_takes_split_keys(const FlashF32Params& p) {
    if (!flash_f32_split_keys_supported(p) || p.lse) return false;
    const long long keys = p.seq_kv ? p.seq_kv : p.seq;
    const bool level = p.mask == kMaskNone && p.dim <= 32 && !flash_f32_split_pays(p);
    return keys >= (level ? kSplitKeysFrom32 : p.dim > 96 ? kSplitKeysFrom128 : kSplitKeysFrom);
}

// Unmasked, head dims 33 to 64, for a forward whose row statistic the gradients read: the gradients' two kernels run side by
// side in one launch (bwd_f32_one_launch) with 128 rows a workgroup, and with 32 would not.  us, forward + gradients, f32 / 128
// rows, B H N at head dim 64: 8 8 256 18.0 + 43.0 / 17.7 + 29.8, 4 8 384 22.3 + 56.7 / 22.5 + 36.8, 2 8 640 32.2 + 86.3 / 32.6 + 51.7,
// 8 16 100 11.3 + 26.6 / 11.9 + 18.9, 1 4 3000 127 + 368 / 129 + 209.  With 32 in one launch as well: 2 8 512 55 / 70, 1 8 1000
// 99 / 125.  The forward alone is level to 0.6 us longer, and inputs that the split does not carry, which the f32 form takes as
// they are, pay for its second pass: 2 8 640 32.3 + 85.7 / 82.2 + 114.4, 8 16 100 12.1 + 27.1 / 17.5 + 33.1.  At head dim 32 the
// forward loses most of what the gradients gain (1 8 2048 50 + 138 / 75 + 109).
static bool flash_f32_gradients_join(const FlashF32Params& p) {
    const long long n_bh = (long long)p.heads * p.batch;
    return p.mask == kMaskNone && p.dim > 32 && p.dim <= 64 && !bwd_f32_one_launch(n_bh * ((p.seq + 31) / 32), 2, p.n_cus) &&
           bwd_f32_one_launch(n_bh * ((p.seq + 127) / 128), 1, p.n_cus);
}

// (above head dim 64 with the row statistic: flash_f32_gradients_wide, flash_bwd_f32.hip)
bool flash_f32_takes_split(const FlashF32Params& p, bool with_lse) {
    if (p.dim % 4 != 0 || p.dim > (with_lse ? 64 : 128) || p.bias || p.mask == kMaskPadding) return false;
    if (with_lse && flash_f32_gradients_join(p)) return true;
    if (p.dim > 64 && p.mask == kMaskNone && !with_lse && flash_f32_takes_split_keys(p)) return flash_f32_rows_pay(p);  // either is ahead of the f32 kernel
    return flash_f32_split_pays(p) && (with_lse || !flash_f32_takes_split_keys(p) || flash_f32_rows_pay(p));
}

hipError_t launch_flash_f32(hipStream_t stream, const FlashF32Params& p) {
    if (p.batch == 0 || p.heads == 0 || p.seq == 0) return hipSuccess;
    dim3 grid((p.seq + kRows - 1) / kRows, p.heads, p.batch), block(64);
    int dt = (p.dim + 31) / 32;
    // the fast kernel reads whole 16-byte chunks: head dim a multiple of 4, rows and bases 16-byte aligned
    auto aligned = [](const void* ptr, const TensorLayout& l) {
        return ((uintptr_t)ptr % 16 == 0) && (l.batch_stride % 4 == 0) && (l.head_stride % 4 == 0) && (l.row_pitch % 4 == 0);
    };
    if (p.dim % 4 == 0 && p.dim <= 128 && aligned(p.q, p.lq) && aligned(p.k, p.lkv) && aligned(p.v, p.lkv) && aligned(p.out, p.lo)) {
        dim3 block4(256);
        FlashF32Params pz = p;
        // 8 (dim <= 64) or 4 waves fit on a CU: is every workgroup resident from the start?
        const long long resident = (long long)p.n_cus * (dt <= 2 ? 2 : 1);
        pz.zigzag = (p.mask == kMaskCausal) && ((long long)grid.x * grid.y * grid.z <= resident) ? 1 : 0;
        deal_to_xcds(pz, grid.x);
        const bool exact = (p.dim % 32 == 0), pad = (p.mask == kMaskPadding);
        if (p.bias && p.mask != kMaskNone) return hipErrorInvalidValue;  // a bias comes without a mask kind
        if (p.lse && flash_f32_gradients_wide(p))  // the statistic of scores formed as the gradients form them
            return flash_f32_rows_pay(p) || !flash_f32_split_keys_supported(p) ? launch_flash_f32_split(stream, p) : launch_flash_f32_split_keys(stream, p);
        if (flash_f32_takes_split(p, p.lse != nullptr)) return launch_flash_f32_split(stream, p);
        if (flash_f32_takes_split_keys(p)) return launch_flash_f32_split_keys(stream, p);
        const int mode = pad ? 2 : (p.mask == kMaskCausal ? 1 : (p.bias ? 3 : 0));
        auto launch = [&](auto dt_c, auto exact_c) {
            constexpr int kDT = decltype(dt_c)::value;
            constexpr bool kEx = decltype(exact_c)::value;
            switch (mode) {
                case 0: hipLaunchKernelGGL((flash_fwd_f32_splitk_kernel<kDT, kEx, 0>), grid, block4, 0, stream, pz); break;
                case 1: hipLaunchKernelGGL((flash_fwd_f32_splitk_kernel<kDT, kEx, 1>), grid, block4, 0, stream, pz); break;
                case 2: hipLaunchKernelGGL((flash_fwd_f32_splitk_kernel<kDT, kEx, 2>), grid, block4, 0, stream, pz); break;
                default: hipLaunchKernelGGL((flash_fwd_f32_splitk_kernel<kDT, kEx, 3>), grid, block4, 0, stream, pz); break;
            }
        };
        auto launch_dt = [&](auto dt_c) {
            if (exact) launch(dt_c, std::true_type{});
            else launch(dt_c, std::false_type{});
        };
        switch (dt) {
            case 1: launch_dt(std::integral_constant<int, 1>{}); break;
            case 2: launch_dt(std::integral_constant<int, 2>{}); break;
            case 3: launch_dt(std::integral_constant<int, 3>{}); break;
            case 4: launch_dt(std::integral_constant<int, 4>{}); break;
            default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }
    if (p.bias || (p.seq_kv && p.seq_kv != p.seq)) return hipErrorInvalidValue;  // only the tiled kernel above does these
    switch (dt) {
        case 1: hipLaunchKernelGGL(flash_fwd_f32_kernel<1>, grid, block, 0, stream, p); break;
        case 2: hipLaunchKernelGGL(flash_fwd_f32_kernel<2>, grid, block, 0, stream, p); break;
        case 3: hipLaunchKernelGGL(flash_fwd_f32_kernel<3>, grid, block, 0, stream, p); break;
        case 4: hipLaunchKernelGGL(flash_fwd_f32_kernel<4>, grid, block, 0, stream, p); break;
        // head dims 129..256: the same kernel with a wider tile (about 100 KB of LDS, one workgroup per CU)
        case 5: hipLaunchKernelGGL(flash_fwd_f32_kernel<5>, grid, block, 0, stream, p); break;
        case 6: hipLaunchKernelGGL(flash_fwd_f32_kernel<6>, grid, block, 0, stream, p); break;
        case 7: hipLaunchKernelGGL(flash_fwd_f32_kernel<7>, grid, block, 0, stream, p); break;
        case 8: hipLaunchKernelGGL(flash_fwd_f32_kernel<8>, grid, block, 0, stream, p); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace rt
