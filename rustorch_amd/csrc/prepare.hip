// The steps between the QKV projection and decode attention, in one launch: per-head RMSNorm of q and k
// (model.rs:862-897, Qwen3 q_norm / k_norm), half-split RoPE (rope.rs:162-205: dim k pairs with dim k + D/2,
// cos/sin from the tables of RoPE::new) and the append of k and v to the caches (llm_kernels.rs:353-372) -- steps
// 2a, 2b and 3 of LlamaModel::decode_step (crates/rustorch-llm/src/model.rs:575-636), for a batch of sequences
// with their own positions and `seq` new tokens each (1 when decoding, the prompt length when prefilling: the
// [batch, heads, seq, head_dim] layout and the position_offset + s rule of rope.rs:92-96, the row range
// [current_len, current_len + seq) of kv_cache.rs:97-110), on bf16 storage.
//
// Every value is widened to f32, run through the reference's f32 arithmetic in the reference's order -- the sum
// of squares is taken sequentially, products and sums are rounded separately (this file is compiled with
// floating-point contraction off) -- and rounded to bf16 once, so the result is the bf16 rounding of what the
// CPU path computes on the same bf16 inputs, bit for bit.
#include <type_traits>

#include "rt_common.hpp"
#include "rt_kernels.hpp"

#pragma clang fp contract(off)

namespace rt {

namespace {

constexpr int kPrepMaxD = 512;

// grid (n_heads + n_kv, seq, batch), one wave per head row; lane l holds the pairs (k, k + D/2), k = l + 64 j, j < PAIRS.  What
// bounds a decode step's launch is its chain of waits, so everything it reads is requested at once (the arguments in one go; then
// the row, gamma and V, which no position is needed for, then the table row) and the one serial part, the sum of squares in index
// order, adds squares that the lanes have formed in parallel, four per LDS read.  The requests go through descriptors: what a lane
// or a head does not have (pairs behind the last, gamma, V beside q) is a zero and no branch.  Where each pair stood behind a test, the
// second waited for the first, and V for the row: in a recorded graph, us a launch, 32 + 8 heads of 128 2.56 -> 2.26, without gamma 1.95 ->
// 1.88, 64 sequences of them 3.43 -> 3.06, 16 + 2 of 256 3.29 -> 2.96.
template <int PAIRS>
__global__ __launch_bounds__(64) void decode_prepare_kernel(DecodePrepareParams p) {
    __shared__ __attribute__((aligned(16))) float squares[2 * PAIRS * kWave];
    const int lane = threadIdx.x;
    const int h = blockIdx.x, sq = blockIdx.y, b = blockIdx.z;
    asm volatile("" ::"s"(p.q), "s"(p.k_in), "s"(p.v_in), "s"(p.k_cache), "s"(p.v_cache), "s"(p.positions), "s"(p.q_gamma), "s"(p.k_gamma), "s"(p.cos_table), "s"(p.sin_table),
                 "s"(p.eps), "s"(p.pos), "s"(p.seq), "s"(p.n_heads), "s"(p.n_kv), "s"(p.head_dim), "s"(p.max_seq), "s"(p.table_rows));
    const int D = p.head_dim, half = D / 2, S = p.seq;
    const bool is_q = h < p.n_heads;
    const int kvh = h - p.n_heads;
    const size_t q_row = (((size_t)b * p.n_heads + h) * S + sq) * D;
    const size_t kv_row = (((size_t)b * p.n_kv + kvh) * S + sq) * D;
    const float* gamma = is_q ? p.q_gamma : p.k_gamma;
    auto rows = [](const void* base, int bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, kBufferFlags); };
    const __amdgpu_buffer_rsrc_t src = rows(is_q ? p.q + q_row : p.k_in + kv_row, 2 * D), gm = rows(gamma, gamma ? 4 * D : 0),
                                 vs = rows(is_q ? p.q : p.v_in + kv_row, is_q ? 0 : 2 * D);
    auto bf16_at = [](__amdgpu_buffer_rsrc_t rs, int k) { return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 2 * k, 0, 0); };
    auto f32_at = [](__amdgpu_buffer_rsrc_t rs, int k) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, 4 * k, 0, 0)); };

    float x0[PAIRS], x1[PAIRS], c[PAIRS], si[PAIRS], g0[PAIRS], g1[PAIRS];
    uint16_t r0[PAIRS], r1[PAIRS], v0[PAIRS], v1[PAIRS];
#pragma unroll
    for (int j = 0; j < PAIRS; j++) {
        const int k = lane + kWave * j;
        r0[j] = bf16_at(src, k);
        r1[j] = bf16_at(src, k + half);
        g0[j] = f32_at(gm, k);
        g1[j] = f32_at(gm, k + half);
        v0[j] = bf16_at(vs, k);
        v1[j] = bf16_at(vs, k + half);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int pos0 = p.positions ? *(const __attribute__((address_space(4))) int32_t*)(p.positions + b) : p.pos;
    // a sequence whose rows would leave the cache or the tables writes nothing (the host checks a scalar position;
    // positions that live on the device are the caller's to keep in range)
    if (pos0 < 0 || pos0 + S > p.max_seq || pos0 + S > p.table_rows) return;
    const int pos = pos0 + sq;
    const size_t cache_row = (((size_t)b * p.n_kv + kvh) * (size_t)p.max_seq + (size_t)pos) * D;
    const __amdgpu_buffer_rsrc_t cs = rows(p.cos_table + (size_t)pos * half, 4 * half), sn = rows(p.sin_table + (size_t)pos * half, 4 * half);
#pragma unroll
    for (int j = 0; j < PAIRS; j++) {
        c[j] = f32_at(cs, lane + kWave * j);
        si[j] = f32_at(sn, lane + kWave * j);
    }
    __builtin_amdgcn_sched_barrier(0);  // (all on their way before the first is awaited)
#pragma unroll
    for (int j = 0; j < PAIRS; j++) {
        x0[j] = bf16_bits_to_f32(r0[j]);
        x1[j] = bf16_bits_to_f32(r1[j]);
    }
    if (gamma) {
        // rms_norm_inplace (model.rs:862-885): sq accumulates in index order; every lane walks the whole row (broadcast
        // reads), which keeps the reference's summation order without a serial section
#pragma unroll
        for (int j = 0; j < PAIRS; j++) {
            const int k = lane + kWave * j;
            if (k >= half) break;
            squares[k] = x0[j] * x0[j];
            squares[k + half] = x1[j] * x1[j];
        }
        __syncthreads();
        float sum = 0.0f;
        int i = 0;
        for (; i + 32 <= D; i += 32) {
            f32x4_t t[8];
#pragma unroll
            for (int e = 0; e < 8; e++) t[e] = *(const f32x4_t*)(squares + i + 4 * e);
#pragma unroll
            for (int e = 0; e < 32; e++) sum = sum + t[e / 4][e % 4];
        }
        for (; i < D; i++) sum = sum + squares[i];
        const float inv_d = 1.0f / (float)D;
        const float inv_rms = 1.0f / sqrtf(sum * inv_d + p.eps);
#pragma unroll
        for (int j = 0; j < PAIRS; j++) {
            x0[j] = x0[j] * inv_rms * g0[j];
            x1[j] = x1[j] * inv_rms * g1[j];
        }
    }
    uint16_t* dst = is_q ? p.q + q_row : p.k_cache + cache_row;
#pragma unroll
    for (int j = 0; j < PAIRS; j++) {
        const int k = lane + kWave * j;
        if (k >= half) break;
        dst[k] = f32_to_bf16_bits(x0[j] * c[j] - x1[j] * si[j]);
        dst[k + half] = f32_to_bf16_bits(x1[j] * c[j] + x0[j] * si[j]);
        if (!is_q) {
            p.v_cache[cache_row + k] = v0[j];
            p.v_cache[cache_row + k + half] = v1[j];
        }
    }
}

// A prompt's rows leave past the caches, with `nt sc1` (at device scope: nothing of them is left in an L2 when the launch ends,
// and nothing is kept there for the rows that come behind), and V, which is only passed through, comes with `nt`.
// B=4, 32 + 8 heads, 4096 tokens, D=128, us with 6 sets of inputs in turn: plain 92.7; rows out `nt` 87.9, `sc1` 89.7,
// `nt sc1` 83.8, V's loads `nt` too 80.3, q's and k's as well 82.8.  (The compiler has a builtin for both bits on buffer stores.)
template <bool kPast>
__device__ __forceinline__ void put16(__amdgpu_buffer_rsrc_t rs, uint32_t byte, u32x4_t v) {
    constexpr int kNt = 2, kSc1 = 16;
    __builtin_amdgcn_raw_buffer_store_b128(v, rs, byte, 0, kPast ? kNt | kSc1 : 0);
}

// The same arithmetic for a prompt.  With many consecutive tokens per head the one-wave kernel above is bound by its
// own redundancy (all 64 lanes of a wave take the same sum of squares, and a row is moved two bytes per lane): 308 us
// for B=4, 32 + 8 heads, 4096 tokens, D=128 (1.3 TB/s; 84 us = 4.8 TB/s here).  A workgroup takes ROWS consecutive tokens of one
// (sequence, head) -- contiguous rows in q / k_in and in the cache -- through LDS: the rows arrive with 16-byte loads,
// every thread takes the sum of squares of ONE row in index order (the reference's order, model.rs:862-885), and
// the normalised, rotated rows leave with 16-byte stores.  Rows sit in LDS as bf16 with a pitch of D + 2 elements (an odd
// number of 32-bit words: the 64 lanes that walk 64 rows in step hit 64 different banks).  D a multiple of 16, at most
// DMAX; every pointer 16-byte aligned.  Grid (token blocks, heads, batch), token blocks fastest: workgroups go round-robin
// to the 8 XCDs in that order, so all heads of a token block run on one XCD and its cos / sin rows are fetched into one
// L2, once (with the heads fastest every XCD fetched every table row: 76 MB more on the prompt above).
// A thread asks for its rows and V at once and for the tables in two halves, the second in the rows' registers: 62 at DMAX 128, so that a
// CU holds eight workgroups (with all tables at once 74, six of them, which 1 x 3000 tokens notice).  One chunk behind the other,
// each with a division ahead of it, and the tables behind the sums: us, 4 x 4096 tokens, 32 / 8 heads of 128 80.3 -> 71.5, without gamma 72.4 ->
// 69.5, 1 x 1000 9.9 -> 8.3, 1 x 100 6.3 -> 5.3; 4 x 16 / 2 of 256, 4096 86.7 -> 66.6.
template <int ROWS, int DMAX, bool kPast>
__global__ __launch_bounds__(256) void prompt_prepare_kernel(DecodePrepareParams p) {
    constexpr int NC = ROWS * DMAX / 8 / 256, NP = NC / 2;  // 16-byte chunks of the rows, and pairs of them, a thread takes
    __shared__ uint32_t rows_w[ROWS * (DMAX + 2) / 2];
    __shared__ float inv[ROWS];
    __shared__ alignas(16) float gam[DMAX];
    const int tid = threadIdx.x;
    const int h = blockIdx.y, b = blockIdx.z;
    asm volatile("" ::"s"(p.q), "s"(p.k_in), "s"(p.v_in), "s"(p.k_cache), "s"(p.v_cache), "s"(p.positions), "s"(p.q_gamma), "s"(p.k_gamma), "s"(p.cos_table), "s"(p.sin_table),
                 "s"(p.eps), "s"(p.pos), "s"(p.seq), "s"(p.n_heads), "s"(p.n_kv), "s"(p.head_dim), "s"(p.max_seq), "s"(p.table_rows), "s"(p.chunk_magic), "s"(p.pair_magic));
    const int sq0 = (int)blockIdx.x * ROWS;
    const int D = p.head_dim, half = D / 2, S = p.seq;
    const int pitch_w = (D + 2) / 2;  // words per row in LDS
    const int CH = D / 8;             // 16-byte chunks per row
    const int HP = half / 8;          // chunk pairs (k .. k + 8, k + half .. k + half + 8) per row
    if (sq0 >= S) return;
    const int n_rows = min(ROWS, S - sq0);
    const bool is_q = h < p.n_heads;
    const int kvh = h - p.n_heads;
    const size_t q_row = (((size_t)b * p.n_heads + h) * S + sq0) * D;
    const size_t kv_row = (((size_t)b * p.n_kv + kvh) * S + sq0) * D;
    const float* gamma = is_q ? p.q_gamma : p.k_gamma;
    const int row_bytes = n_rows * D * 2;
    auto rsrc = [](const void* base, int bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, kBufferFlags); };
    const __amdgpu_buffer_rsrc_t src = rsrc(is_q ? p.q + q_row : p.k_in + kv_row, row_bytes), gm = rsrc(gamma, gamma ? 4 * D : 0),
                                 vs = rsrc(is_q ? p.q : p.v_in + kv_row, is_q ? 0 : row_bytes);
    u32x4_t x[NC], v[NC];  // chunk c = tid + 256 i of the block's rows, which follow one another
#pragma unroll
    for (int i = 0; i < NC; i++) x[i] = __builtin_amdgcn_raw_buffer_load_b128(src, 16 * (tid + 256 * i), 0, 0);
    const float g = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(gm, 4 * tid, 0, 0));
#pragma unroll
    for (int i = 0; i < NC; i++) v[i] = __builtin_amdgcn_raw_buffer_load_b128(vs, 16 * (tid + 256 * i), 0, kPast ? 2 : 0);
    __builtin_amdgcn_sched_barrier(0);
    const int pos0 = p.positions ? *(const __attribute__((address_space(4))) int32_t*)(p.positions + b) : p.pos;
    if (pos0 < 0 || pos0 + S > p.max_seq || pos0 + S > p.table_rows) return;  // as in the one-wave kernel
    const size_t table_row = (size_t)(pos0 + sq0) * half, cache_row = (((size_t)b * p.n_kv + kvh) * (size_t)p.max_seq + (size_t)(pos0 + sq0)) * D;
    const __amdgpu_buffer_rsrc_t cs = rsrc(p.cos_table + table_row, row_bytes), sn = rsrc(p.sin_table + table_row, row_bytes);  // (half as many, twice as wide)
    f32x4_t ct[NP][2], st[NP][2];  // of pair c = tid + 256 i: eight values of each table, which follow one another likewise
    auto tables = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            ct[i][e] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(cs, 32 * (tid + 256 * i) + 16 * e, 0, 0));
            st[i][e] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(sn, 32 * (tid + 256 * i) + 16 * e, 0, 0));
        }
    };
#pragma unroll
    for (int i = 0; i < NP / 2; i++) tables(i);
    __builtin_amdgcn_sched_barrier(0);  // (all on their way before the first is awaited)

#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = tid + 256 * i;
        if (c >= n_rows * CH) break;
        const int r = (int)(((uint32_t)c * p.chunk_magic) >> 20), ch = c - r * CH;
        uint32_t* w = rows_w + r * pitch_w + 4 * ch;  // (rows start on odd words: four 4-byte writes)
        w[0] = x[i][0];
        w[1] = x[i][1];
        w[2] = x[i][2];
        w[3] = x[i][3];
    }
    if (tid < DMAX) gam[tid] = g;
    __builtin_amdgcn_sched_barrier(0);  // (these in the rows' registers)
#pragma unroll
    for (int i = NP / 2; i < NP; i++) tables(i);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    if (!is_q) {
        const __amdgpu_buffer_rsrc_t vd = rsrc(p.v_cache + cache_row, row_bytes);
#pragma unroll
        for (int i = 0; i < NC; i++) put16<kPast>(vd, 16u * (uint32_t)(tid + 256 * i), v[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (gamma) {
        for (int r = tid; r < n_rows; r += 256) {
            const uint32_t* w = rows_w + r * pitch_w;
            float sq = 0.0f;
            for (int j = 0; j < half; j++) {  // elements 2j and 2j + 1, in index order
                const uint32_t y = w[j];
                const float v0 = bf16_lo(y), v1 = bf16_hi(y);
                sq = sq + v0 * v0;
                sq = sq + v1 * v1;
            }
            const float inv_d = 1.0f / (float)D;
            inv[r] = 1.0f / sqrtf(sq * inv_d + p.eps);
        }
    }
    if (gamma) __syncthreads();
    const __amdgpu_buffer_rsrc_t dst = rsrc(is_q ? p.q + q_row : p.k_cache + cache_row, row_bytes);
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int c = tid + 256 * i;
        if (c >= n_rows * HP) break;
        const int r = (int)(((uint32_t)c * p.pair_magic) >> 20), k0 = 8 * (c - r * HP);
        const uint32_t* w = rows_w + r * pitch_w;
        float x0[8], x1[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t y = w[k0 / 2 + e], z = w[(half + k0) / 2 + e];
            x0[2 * e] = bf16_lo(y);
            x0[2 * e + 1] = bf16_hi(y);
            x1[2 * e] = bf16_lo(z);
            x1[2 * e + 1] = bf16_hi(z);
        }
        if (gamma) {
            const float inv_rms = inv[r];
            auto times = [&](float (&y)[8], const float* at) __attribute__((always_inline)) {
                const f32x4_t ga = *(const f32x4_t*)at, gb = *(const f32x4_t*)(at + 4);
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] = y[e] * inv_rms * (e < 4 ? ga[e] : gb[e - 4]);
            };
            times(x0, gam + k0);
            __builtin_amdgcn_sched_barrier(0);
            times(x1, gam + half + k0);
        }
        u32x4_t o0, o1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int i0 = 2 * e, i1 = 2 * e + 1;
            const float c0 = ct[i][i0 / 4][i0 % 4], c1 = ct[i][i1 / 4][i1 % 4], s0 = st[i][i0 / 4][i0 % 4], s1 = st[i][i1 / 4][i1 % 4];
            o0[e] = pack_bf16x2(x0[i0] * c0 - x1[i0] * s0, x0[i1] * c1 - x1[i1] * s1);
            o1[e] = pack_bf16x2(x1[i0] * c0 + x0[i0] * s0, x1[i1] * c1 + x0[i1] * s1);
        }
        put16<kPast>(dst, (uint32_t)(r * D + k0) * 2u, o0);
        put16<kPast>(dst, (uint32_t)(r * D + half + k0) * 2u, o1);
        __builtin_amdgcn_sched_barrier(0);
    }
}

bool aligned16(const void* a) { return ((uintptr_t)a & 15) == 0; }

}  // namespace

hipError_t launch_decode_prepare(hipStream_t stream, const DecodePrepareParams& p) {
    if (p.batch == 0 || p.seq == 0 || p.n_heads + p.n_kv == 0 || p.head_dim == 0) return hipSuccess;
    if (p.head_dim > kPrepMaxD || (p.head_dim & 1) || p.seq > 65535 || p.batch > 65535) return hipErrorInvalidValue;
    // a prompt: the kernel that moves 64 or 128 consecutive tokens of a head through LDS, where its loads and stores are whole
    // 16-byte chunks (64 rows: 17 or 33 KB of LDS, so that four to eight workgroups share a CU; with 256 rows the same
    // prompt took 113 us instead of 80)
    const bool wide_ok = p.seq >= 32 && p.head_dim % 16 == 0 && p.head_dim <= 256 && aligned16(p.q) && aligned16(p.k_in) &&
                         aligned16(p.v_in) && aligned16(p.k_cache) && aligned16(p.v_cache) && aligned16(p.cos_table) &&
                         aligned16(p.sin_table) && aligned16(p.q_gamma) && aligned16(p.k_gamma) && p.n_heads + p.n_kv <= 65535;
    if (wide_ok) {
        // past the caches from twice what the L2s hold, 8 of 4 MB.  us, plainly / past, buffers of four calls in turn, and the copies that
        // bring the inputs and the call together, 32 / 8 heads of 128: 1 x 4096 tokens (50 MB) 18.1 / 22.6, 35.4 / 35.3; 1 x 4500 (55) 23.5 / 25.2,
        // 38.9 / 39.1; 1 x 5000 (61) 28.0 / 27.1, 42.2 / 42.0; 1 x 5500 (68) 30.4 / 29.0, 46.1 / 45.6; 2 x 3000 (74) 33.2 / 31.5, 50.9 / 49.9; 2 x 3500
        // (86) 38.9 / 35.6, 62.6 / 56.1; 16 x 512 (101) 44.1 / 39.0, 85.2 / 63.8; 4 x 4096 (201) 79.0 / 72.0; 8 x 16 / 16 of 64, 1300 (64) 35.6 / 32.0,
        // 45.0 / 44.1; of 256, 4 x 8 / 8, 1300 (64) 35.0 / 30.3, 46.8 / 45.8, 4 x 16 / 2, 3500 (143) 64.8 / 59.5, 110.1 / 107.9.  Inputs that still lie in the
        // last-level cache favour plain rows: 1 x 5500 27.9 / 29.2, 2 x 3000 31.3 / 31.4 behind other calls' copies, and a call repeated on one set of
        // buffers, which no prompt is, 23.0 / 28.2, 25.0 / 30.8, 16 x 512 32.1 / 38.4
        const double written = 2.0 * p.batch * p.seq * (double)p.head_dim * (p.n_heads + 2.0 * p.n_kv);
        const bool past = written > 64.0 * (1 << 20);
        DecodePrepareParams pp = p;
        pp.chunk_magic = (1u << 20) / (uint32_t)(p.head_dim / 8) + 1u;  // (exact: c d < 2^20)
        pp.pair_magic = (1u << 20) / (uint32_t)(p.head_dim / 16) + 1u;
        auto launch = [&](auto rows_c, auto dmax_c) {
            constexpr int kRows = decltype(rows_c)::value, kDMax = decltype(dmax_c)::value;
            // Token blocks up to a multiple of eight, so that every head's land on the XCD that has their table rows (those behind the last
            // token end at once), where that adds a twelfth at most and rows stay in the caches.  us, as they are / so, four or more sets of buffers in turn, 32 / 8
            // heads of 128: 1 x 4500 tokens (71 blocks) 27.2 / 25.9, 5300 (83) 33.5 / 30.7, 3500 (55) 20.4 / 20.2; but 1 x 2200 (35) 11.0 / 11.5, 2 x 2600
            // (41) 28.4 / 31.3, 4 x 1300 (21) 28.9 / 32.1; past the caches 8 x 1300 46.7 / 52.3, 4 x 2711 (43) 48.4 / 51.8, 2 x 32 / 32 of 80, 2600 46.8 / 53.0, 2 x 5500
            // (86) 49.4 / 50.0.
            int blocks = (p.seq + kRows - 1) / kRows;
            const int eights = (blocks + 7) / 8 * 8;
            if (!past && 12 * (eights - blocks) <= blocks) blocks = eights;
            const dim3 grid(blocks, p.n_heads + p.n_kv, p.batch), block(256);
            if (past) hipLaunchKernelGGL((prompt_prepare_kernel<kRows, kDMax, true>), grid, block, 0, stream, pp);
            else hipLaunchKernelGGL((prompt_prepare_kernel<kRows, kDMax, false>), grid, block, 0, stream, pp);
        };
        // A thread asks for as many chunks as its widest row needs: narrow heads have a form of their own, or half and three quarters of those
        // requests are for nothing.  us, chunks in a loop (before) / rows of up to 128 / of up to 64 / 128 rows of up to 32, recorded: 3 x 16 / 16 heads of 64,
        // 6807 tokens 50.2 / 56.1 / 47.2, 1 x 32 / 8, 1000 5.9 / 5.6 / 5.1, without gamma 4.9 / 4.7 / 4.2; of 48, 2 x 32 / 8, 3000 14.0 / 15.0 / 13.1; of 32, 3 x
        // 16 / 16, 6807 31.9 / 38.0 / 30.0 / 27.0, 4 x 16 / 16, 700 without gamma 6.0 / 6.7 / 5.6 / 4.9, 1 x 32 / 8, 100 3.49 / 3.35 / 3.16 / 3.37.  (128 rows of up to
        // 64: 49.1 and 6.0 us on the first two, 256 of up to 32 30.7 on the fourth.)
        if (p.head_dim <= 32) launch(std::integral_constant<int, 128>{}, std::integral_constant<int, 32>{});
        else if (p.head_dim <= 64) launch(std::integral_constant<int, 64>{}, std::integral_constant<int, 64>{});
        else if (p.head_dim <= 128) launch(std::integral_constant<int, 64>{}, std::integral_constant<int, 128>{});
        else launch(std::integral_constant<int, 64>{}, std::integral_constant<int, 256>{});
        return hipGetLastError();
    }
    const dim3 grid(p.n_heads + p.n_kv, p.seq, p.batch), block(64);
    if (p.head_dim <= 2 * kWave) hipLaunchKernelGGL(decode_prepare_kernel<1>, grid, block, 0, stream, p);
    else if (p.head_dim <= 4 * kWave) hipLaunchKernelGGL(decode_prepare_kernel<2>, grid, block, 0, stream, p);
    else hipLaunchKernelGGL(decode_prepare_kernel<kPrepMaxD / 2 / kWave>, grid, block, 0, stream, p);
    return hipGetLastError();
}

}  // namespace rt
