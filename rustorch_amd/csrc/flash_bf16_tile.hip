// bf16 flash-attention forward for gfx950, the general form: any head dim up to 256 that is a multiple of 8,
// own key count (cross-attention), per-sequence query and key counts (padded batches, chunked decode over a
// cache), causal masks aligned to the last key, the key-padding vector, an additive f32 score bias, and query
// rows that run over (position, head of a GQA group) so that a handful of new positions still fills a tile.
// Device counterpart of flash_forward_masked (crates/rustorch-attention/src/cpu_forward.rs:193-425) for bf16
// tensors: bf16 in, f32 accumulation on the matrix cores, bf16 out rounded once.
//
// Where the 8-wave persistent kernel of flash_bf16.hip hand-schedules two waves per SIMD around one long job
// list, this one is built for many short jobs: a workgroup of four waves owns 128 query rows (32 per wave) of one
// (batch, head) and is gone when they are done; several workgroups share a CU, so one workgroup's set-up, softmax
// and output overlap with another's matrix work without any hand-written interleaving, and the hardware
// dispatcher balances jobs of unequal length.  Keys are walked KT at a time through a double-buffered LDS tile (straight
// from memory, or through registers above head dim 128 and under a key-padding vector whose bits do not fit LDS; one
// workgroup barrier per tile); per 32-key item a wave computes
//
//   S^T[kv, q]  = K[kv, :] . Q[q, :]      v_mfma_f32_32x32x16_bf16, A = K tile (LDS), B = Q (registers)
//   online softmax on S^T (a lane holds 16 scores of query row lane % 32; row max / sum are in-lane plus one
//                          exchange with lane ^ 32)
//   O^T[d, q]  += V^T[d, kv] . P^T[kv, q]  A = V tile read transposed (ds_read_b64_tr_b16), B = P (registers)
//
// with P fed to the second product straight from the score registers (the accumulator layout of the first
// product is a B operand of the second under a fixed permutation of the contraction slots, which the V operand
// read applies as well).  LDS rows are padded, or their 16-byte slots XORed with bits of the row, so that the 16-byte K
// reads and the transposing V reads are free of bank conflicts.
#include "flash_tile_lds.hpp"
#include "rt_common.hpp"
#include "rt_kernels.hpp"

#include <type_traits>

namespace rt {

namespace {

constexpr int TROWS = 128;  // query rows per workgroup: four waves' worth, each wave 32
constexpr float kTileTrigSum = 65536.0f;  // a lane's 16-key share of a row sum above this sends the wave to the slow path

typedef short s16x4t __attribute__((ext_vector_type(4)));
typedef float f32x2t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t t_cvt_pk_bf16(float lo, float hi) {
    f32x2t x = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2t));  // v_cvt_pk_bf16_f32, RNE
}
// Transposing LDS read: within each group of 16 lanes, lane j receives element (j % 4) of the 8 bytes addressed
// by lanes 4e + j/4, e = 0..3.
__device__ __forceinline__ u32x2_t t_lds_read_tr16(const uint16_t* p) {
    s16x4t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4t __attribute__((address_space(3)))*)(p));
    return __builtin_bit_cast(u32x2_t, v);
}
__device__ __forceinline__ float t_vmax(float a, float b) {  // plain v_max_f32: returns the non-NaN operand
    float d;
    asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
    return d;
}
__device__ __forceinline__ float t_max_with_other_half(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return t_vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float t_sum_with_other_half(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Max of the 16 scores a lane holds, as three chains of three-input maxima.  Written with the compiler's own max
// (not inline assembly): the scores come straight out of a matrix instruction, and a vector instruction that reads
// a matrix result needs wait states only the compiler's hazard pass inserts -- it does not look inside assembly.
__device__ __forceinline__ float t_max3(float a, float b, float c) { return __builtin_fmaxf(__builtin_fmaxf(a, b), c); }
__device__ __forceinline__ float t_max16(const f32x16_t& s) {
    float t0 = t_max3(s[0], s[1], s[2]), t1 = t_max3(s[3], s[4], s[5]), t2 = t_max3(s[6], s[7], s[8]);
    t0 = t_max3(t0, s[9], s[10]);
    t1 = t_max3(t1, s[11], s[12]);
    t2 = t_max3(t2, s[13], s[14]);
    return __builtin_fmaxf(t_max3(t0, t1, t2), s[15]);
}

template <int DP, bool DIRECT = false>
struct TileCfg {
    static constexpr int KT = DP > 128 && !DIRECT ? 32 : TileLds<DP>::KT;  // keys per LDS tile
    static constexpr int NI = KT / 32;              // 32-key items per tile
    static constexpr int THREADS = 256;
    static constexpr int LDK = DP + 8;                        // +16 B: 16 rows x 16 B tile all 64 banks
    static constexpr int LDV = DP + (DP % 64 == 0 ? 32 : 0);  // row pitch = 16 or 48 (mod 64) words: 4 rows x 64 B tile all banks
    static constexpr int OCC = DP <= 64 ? 3 : (DP <= 128 ? 2 : 1);  // workgroups per CU the register budget is set for
    static constexpr int DT = DP / 32;
    static constexpr int PF = DP <= 32 ? 2 : 1;  // register sets of tiles in flight (wider rows take too many registers for more)
    static constexpr int TILE_BYTES = 2 * KT * (LDK + LDV) * 2;           // two stages of K and V
    static constexpr int REGION = 32 * LDK * 2;                           // a wave's staged output rows
    static constexpr int LDS_BYTES = TILE_BYTES > 4 * REGION ? TILE_BYTES : 4 * REGION;
    // DIRECT: unpadded tiles (rows of DP * 2 bytes, 16-byte slots swizzled), filled by loads that go straight to LDS
    static constexpr int STAGE_BYTES = TileLds<DP>::STAGE_BYTES;
    static constexpr int LDS_BYTES_DIRECT = 4 * STAGE_BYTES > 4 * REGION ? 4 * STAGE_BYTES : 4 * REGION;
    static constexpr int OCC_DIRECT = OCC;
    static constexpr int BIAS_BYTES = 32 * 32 * 4;  // a wave's bias values of an item: 32 rows of 32 keys
};

// Where a workgroup works that takes the `pos`-th of the query tiles of `batch` <= 64 sequences, ordered by tile number downwards
// (tile L of every sequence that has one, by sequence), then those of padded rows only, by tile number upwards.  Lane i holds
// sequence i: a ballot per tile number gives the sequences that have it, four numbers without a branch between.  It stands
// ahead of the first request for keys, so what bounds it is its own latency: a binary search over the number, a sum over the
// lanes a step, took 0.3 to 1 us more of a launch (below).
struct TilePlace {
    int b, qtile, len;
};
__device__ __forceinline__ TilePlace t_place_by_length(const int32_t* lens, int batch, int seq, int pos, int lane) {
    const int len = lane < batch ? min(max(lens[lane], 0), seq) : 0;
    const int n_all = (seq + TROWS - 1) / TROWS;
    const uint32_t n = (uint32_t)(len + TROWS - 1) / TROWS;                    // its tiles with valid rows,
    const uint32_t m = lane < batch ? (uint32_t)n_all - n : 0u;                // and the others: the last m of n_all
    int at = pos, k = 0;  // k: tiles passed by, of n_all with valid rows (from the highest down) and n_all without
    uint64_t has = 0;
    auto find = [&](auto with) __attribute__((always_inline)) {  // with(k): the sequences that have the k-th; true when the place is among them
        for (k = 0; k < n_all; k += 4) {
            int c[4];
#pragma unroll
            for (int j = 0; j < 4; j++) c[j] = __builtin_popcountll(with(k + j));
            const int all = c[0] + c[1] + c[2] + c[3];
            if (at < all) {
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    if (at < c[j]) break;
                    at -= c[j];
                    k++;
                }
                has = with(k);
                return true;
            }
            at -= all;
        }
        return false;
    };
    int tile;
    if (find([&](int i) __attribute__((always_inline)) { return __ballot((uint32_t)(n_all - 1 - i) < n); })) {  // (below tile 0: none)
        tile = n_all - 1 - k;
    } else {
        find([&](int i) __attribute__((always_inline)) { return __ballot((uint32_t)(n_all - 1 - i) < m); });
        tile = k;
    }
    const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
    const uint64_t one = has & __ballot(below == at);
    const int b = one ? __builtin_ctzll(one) : 0;
    return TilePlace{b, tile, __builtin_amdgcn_readlane(len, b)};
}

// How K/V tiles come into LDS: through registers, or straight there with rows of DP columns or with rows of fewer.
enum TileWay : int { kTilesRegs = 0, kTilesDirect = 1, kTilesDirectPart = 2 };

// MODE: kMaskNone, kMaskCausal, kMaskPadding.  BIAS: an additive f32 score bias is applied (then MODE is kMaskNone).
// PACKED: query rows run over (position, head of the GQA group) (then MODE is kMaskCausal and there is no bias).
// The grid is (heads or kv heads, batch, query tiles): no division stands between a workgroup and its first load.
//
// The key walk of a wave is a software pipeline over 32-key items, one step per item j:
//
//   S(j+1) = K(j+1).Q^T           KS matrix instructions   | both independent of the vector work, issued in between
//   O^T   += V(j-1)^T.P(j-1)^T    2 DT matrix instructions | it so that the wave never waits on the matrix pipe
//   P(j)   = softmax step on S(j)  ~60 vector instructions
//
// so a wave that is alone on its SIMD (the long query tiles at the end of a launch of short sequences) keeps the
// matrix pipe and the vector pipe busy at once instead of running the three phases of an item back to back.
// K therefore sits in LDS one tile ahead of V: during tile t the waves read K(t+1) and V(t-1), and after the
// tile's one barrier (behind the step of its first item) K(t+2) and V(t+1) are parked over K(t) and V(t-1).
//
// SPLIT (packed rows only): the keys of a (sequence, kv head) are cut into p.n_splits spans of whole tiles, a
// workgroup walks one span and leaves the unnormalised O, the running max and the row sum of its rows as a partial
// (o, m, l); flash_split_merge_kernel folds the partials with the online-softmax monoid
// (crates/rustorch-attention/src/online_softmax.rs:105-131 extended with o) -- the split over the context of the
// decode kernels, for a chunk of new positions over one long cache, whose few query tiles would otherwise keep a
// handful of CUs busy.
//
// WIN (causal mask, rows of one head): a sliding window, query i sees keys (i + off - window, i + off] -- the
// reference's sliding_window_mask (crates/rustorch-nn/src/masks.rs:41-60) without its [T, T] bias tensor.  The walk
// starts at the tile that holds the first key the workgroup's first row sees (tensor base, key count and causal offset
// moved by that many keys, as for a span of SPLIT), and an item that holds keys below some row's window is masked on
// that side as well.
//
// DIRECT: the tiles travel from memory straight into LDS
// (buffer_load_dwordx4 ... lds) instead of through registers and LDS writes.  After a tile's barrier the waves request
// K(t+2) and V(t+1) into the stages K(t) and V(t-1) have just left and wait for their own requests ahead of the next
// tile's barrier.  LDS rows are unpadded (a landing block of 1 KB is contiguous) and their 16-byte slots are XORed
// with bits of the row, as in flash_bf16.hip.  Same instructions on the same operands otherwise: the same bits.
// Measured against the register path, interleaved in one process: 3-5 % on short or padded sequences (B=16 H=16
// N=1024: 52.3 -> 49.3 us), 7-9 % on long ones (B=4 H=32 N=4096: 306 -> 283 us), 4-7 % at head dim 128, 10-11 % at 96 and
// 80 (B=2 H=16 N=4096: 123.5 -> 111.8 and 119.6 -> 107.7), 5 % at 32 (58.4 -> 55.8), 20-40 % at 256 (takes_tiles_direct), where it
// is what leaves the registers for the pipelined walk: 512 of them, a wave a SIMD; three stages per matrix or four
// workgroups per CU (head dim 64) are no faster.  Head dims between the tile widths have a form of their own
// (kTilesDirectPart), whose requests leave the lanes behind the head dim out: two scalar instructions a request, which
// cost the masked form at head dim 64 6 % where the kernel of whole rows had them too (28.3 -> 29.9 us; a branch 31.1).
//
// HALVES (DIRECT, rows of one head, no window): the workgroup is eight waves, two to a SIMD, and the tiles of its walk are
// cut in two: waves 0-3 take the first half of them and waves 4-7 the second, each half in stages of its own and for the
// same query rows; at the end the second half's O, max and row sum go through LDS to the first, which folds them in as
// the split form's merge does.  For launches that leave a CU one workgroup: its waves, alone on their SIMDs, take 800
// clocks an item at head dim 64 where three of them together take 500 each, and 2100 with a bias, whose latency one wave
// does not hide.  (launch_halves has the figures.)
template <int DP, int MODE, bool BIAS, bool PACKED, bool SPLIT = false, bool WIN = false, int TILES = kTilesRegs, bool HALVES = false, bool QROWS = true, bool PAST = false>
__global__ __launch_bounds__(HALVES ? 512 : TileCfg<DP>::THREADS, HALVES ? 2 : BIAS && DP == 64 ? 2 : (TILES ? TileCfg<DP>::OCC_DIRECT : TileCfg<DP>::OCC)) void flash_tile_bf16_kernel(FlashTileParams p) {
    static_assert(!SPLIT || (PACKED && !BIAS && MODE == kMaskCausal), "the split over the keys serves the chunked decode");
    static_assert(!WIN || (!PACKED && !BIAS && !SPLIT && MODE == kMaskCausal), "the window is a causal mask's");
    static_assert(!HALVES || (TILES != kTilesRegs && !PACKED && !SPLIT && !WIN), "halves of the walk: tiles straight to LDS, rows of one head");
    constexpr bool DIRECT = TILES != kTilesRegs, WHOLE = TILES == kTilesDirect;
    using Cfg = TileCfg<DP, DIRECT>;
    constexpr int KT = Cfg::KT, LDK = Cfg::LDK, LDV = Cfg::LDV, NI = Cfg::NI, TTHREADS = Cfg::THREADS;
    constexpr int KS = DP / 16;        // contraction steps of the score product
    constexpr int DT = DP / 32;        // 32-row tiles of O^T
    constexpr int NM = 2 * KS;         // matrix instructions of a step: KS for S(j+1), 2 DT = KS for P(j-1).V(j-1)
    constexpr int CH = DP / 8;         // 16-byte chunks per (padded) row
    constexpr int CHUNKS = KT * CH;    // chunks of one matrix's tile
    constexpr int NL = (CHUNKS + TTHREADS - 1) / TTHREADS;  // chunks a thread moves per matrix per tile
    constexpr bool kCausal = MODE == kMaskCausal;
    constexpr int PF = Cfg::PF;        // register sets of tiles in flight behind the two LDS stages
    static_assert(2 * DT == KS, "one P.V matrix instruction per score matrix instruction");
    // Through registers, head dims above 128 do not have those for two score tiles and their operands in flight beside the tiles'
    // own (O alone is 128, and a wave has a SIMD to itself), nor does head dim 128 with a key-padding mask: there an item runs its
    // three phases one after the other, and K is parked with V.
    constexpr bool PIPE = DIRECT || DP < 128 || (DP == 128 && MODE != kMaskPadding);
    static_assert(!BIAS || (DP <= 128) == DIRECT, "a bias comes with tiles straight to LDS up to head dim 128, through registers above");
    static_assert(PIPE || !HALVES, "the halves meet once a tile");

    // QLDS: the query rows come through LDS as well, whole lines an instruction, over V(1), whose request comes behind the first
    // barrier only, and as many bytes behind it.  Read straight into the operands, 16 bytes of 32 rows at a time, every line was
    // asked for by four instructions (eight at head dim 128).  us, inputs that change from pass to pass, bhnd / bnhd, before ->
    // now: window 256, 4 16 4096 64 43.9 -> 42.5 / 47.0 -> 45.2, window 64 34.2 -> 32.9 / 37.0 -> 34.8, window 126, 5 12 7697 128
    // 113.2 -> 107.6 / 120.2 -> 112.8; causal 2 32/8 1501 128 46.3 -> 45.3 / 46.7 -> 45.8, 4 16 1024 64 16.7 -> 16.4; masked 4 16
    // 1024 64 31.2 -> 30.5.  Past the caches as well under a window up to head dim 64 where the
    // workgroups do not fit the chip at once (42.7 -> 41.4 / 45.5 -> 45.2; 1 8/2 852 64 window 104 7.7 -> 7.8); elsewhere that is
    // slower (causal 2 32/8 1501 128 45.2 -> 47.4).  Not where rows run over a group's heads, nor up to head dim 32, whose rows are half
    // a line (2 32 3000 32 window 500 26.9 -> 27.3), nor beside a bias at head dim 128, where two workgroups a CU would not fit, or up to
    // 64 (QROWS) where a third one would be there: masked 9 16 1261 x 309 64 39.5 -> 42.0, 6 16 900 x 200 15.7 -> 16.7.
    constexpr bool QLDS = DIRECT && !PACKED && !(BIAS && DP == 128) && (DP > 32 || MODE == kMaskPadding) && QROWS;
    static_assert(!QLDS || KT * 2 == TROWS, "half of the query rows fit a stage");
    constexpr int kTilesLds = QLDS ? (5 * Cfg::STAGE_BYTES > 4 * Cfg::REGION ? 5 * Cfg::STAGE_BYTES : 4 * Cfg::REGION) : DIRECT ? Cfg::LDS_BYTES_DIRECT : Cfg::LDS_BYTES;  // BIAS: the four waves' bias values behind the tiles
    constexpr int kHalves = HALVES ? 2 : 1, kBiasAt = kHalves * ((kTilesLds + 1023) / 1024 * 1024);
    static_assert(!HALVES || (kTilesLds % 1024 == 0 && kTilesLds >= 4 * 32 * DP * 4 && kTilesLds >= 4 * Cfg::REGION + 2048), "a half's partials fit over its tiles, their max and sum behind the output rows");
    __shared__ alignas(DIRECT || BIAS ? 1024 : 16) unsigned char lds[BIAS ? kBiasAt + kHalves * 4 * Cfg::BIAS_BYTES : kHalves * kTilesLds];
    uint16_t* const Ks = (uint16_t*)lds;                      // [2][KT * LDK]
    uint16_t* const Vs = (uint16_t*)lds + 2 * KT * LDK;       // [2][KT * LDV]
    using Lds = TileLds<DP>;  // DIRECT
    constexpr int ROWB = Lds::ROW_BYTES, STAGE_B = Lds::STAGE_BYTES;

    const int tid = HALVES ? threadIdx.x & 255 : threadIdx.x;  // within the half
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = HALVES ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const uint32_t half_at = (uint32_t)(half * kTilesLds);  // where its stages start
    const int col = lane & 31, hh = lane >> 5;

    // ---- which tile.  The grid is (unit within the batch, batch, rank of the query tile), dispatched x first: all
    // units' tiles of rank 0 (the last query tile, the longest causal rows), then rank 1, ... -- the dispatcher hands a
    // free slot the next tile in that order, so the long ones start first and the short ones fill the gaps at the
    // end.  Workgroups go round-robin to the 8 XCDs (each with its own L2) in the same order: when the units
    // ((batch, head) pairs, or (batch, kv head) when rows are packed) divide by 8, all query tiles of a unit land on
    // one XCD and share K and V through its L2.
    const int G = PACKED ? p.pack : 1;  // heads per packed row block (1: rows are positions of one head)
    const int rows_total = p.seq_q * G;
    // The heads of a GQA group follow one another at a distance of kv_heads in the grid, so that a group lands on one XCD
    // (or on those its kv heads leave it) and shares its keys through that L2: grid position x is head x / kv_heads of
    // group x % kv_heads (kv_magic = 2^32 / kv_heads + 1, exact below 2^16 heads; 0 where every head has its own keys).
    int b = blockIdx.y;
    const int gx = PACKED ? 0 : (int)__umulhi(blockIdx.x, p.kv_magic);
    const int kvh = (int)blockIdx.x - gx * p.kv_heads;
    const int hx = PACKED ? kvh : kvh * p.group + gx;
    const int zz = p.n_qtiles - 1 - (int)blockIdx.z;
    // A padded batch by length (n_qtiles < 0, tiles_by_length): the position within (batch, rank) is a place in the list of
    // all sequences' query tiles by their number, which is their cost: the last tile of the longest sequence first, the tiles
    // of padded rows only last.  Ranked within their own sequence, the second and third tile of the longest one waited behind
    // first tiles of short ones.
    constexpr bool kByLength = kCausal && !PACKED && !SPLIT && !WIN;
    TilePlace place{-1, 0, 0};
    // (what the first requests need of the arguments is loaded ahead of the branch, not once more behind it)
    if (kByLength) asm volatile("" ::"s"(p.k), "s"(p.v), "s"(p.lkv.batch_stride), "s"(p.lkv.head_stride), "s"(p.lkv.row_pitch), "s"(p.seq_kv), "s"(p.dim));
    if (kByLength && p.n_qtiles < 0) {
        place = t_place_by_length(p.q_lens, (int)gridDim.y, p.seq_q, (int)(blockIdx.y + gridDim.y * blockIdx.z), lane);
        b = place.b;
    }
    const int h0 = PACKED ? hx * G : hx;  // head of a row with g = 0
    const int D = p.dim;

    const uint16_t* __restrict__ Kg = p.k + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    const uint16_t* __restrict__ Vg = p.v + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;

    // ---- tile movement: chunk c = tid + TTHREADS n of a tile is (row c / CH, 16-byte chunk c % CH).  A tile
    // travels global -> registers -> LDS.  LDS holds two stages of each matrix; PF register sets per matrix hold
    // the tiles behind them, so that a load has PF tile-times to arrive.
    u32x4_t kreg[PF][NL], vreg[PF][NL];
    uint32_t keep_raw[PF];
#pragma unroll
    for (int i = 0; i < PF; i++) {
        keep_raw[i] = 1;
#pragma unroll
        for (int n = 0; n < NL; n++) kreg[i][n] = vreg[i][n] = u32x4_t{0u, 0u, 0u, 0u};  // (only read when there are no keys at all)
    }
    // per-thread constants of the movement (hoisted: the loop then spends a handful of instructions per tile on it)
    uint32_t ld_off[NL];  // byte offset of the thread's chunk from the first byte of a tile; the same in K and V
    uint32_t st_k[NL], st_v[NL];  // byte offsets of the chunk in an LDS stage
    bool ld_on[NL];
    const uint32_t kv_pitch = (uint32_t)p.lkv.row_pitch;
#pragma unroll
    for (int n = 0; n < NL; n++) {
        const int c = tid + TTHREADS * n;
        const int row = c / CH, ch = c - row * CH;
        st_k[n] = (uint32_t)((row * LDK + 8 * ch) * 2);
        st_v[n] = (uint32_t)((2 * KT * LDK + row * LDV + 8 * ch) * 2);
        ld_on[n] = 8 * ch < D;
        // a chunk past the head dim is requested (from column 0) but never parked
        ld_off[n] = ((uint32_t)row * kv_pitch + (ld_on[n] ? (uint32_t)(8 * ch) : 0u)) * 2u;
    }
    u32x4_t k1[NL];
    // DIRECT: which chunk of a tile each lane of a load instruction fetches, and where it lands (flash_tile_lds.hpp).  Slots
    // behind the head dim are not requested.
    constexpr int SPR = Lds::SPR, NLD = Lds::REQUESTS;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    int dl_row[NLD];                            // row of the lane's chunk of instruction n,
    uint32_t dl_k[NLD], dl_v[NLD];              // its byte offsets from a tile's first row in K and in V,
    uint64_t dl_k_on[NLD], dl_v_on[NLD];        // and the lanes whose chunk lies within the head dim
#pragma unroll
    for (int n = 0; n < NLD; n++) {
        const int c = 64 * (wave + 4 * n) + lane, row = (int)((uint32_t)c / SPR), slot = c - row * SPR;
        dl_row[n] = row;
        const int sk = slot ^ Lds::swz_k(row), sv = slot ^ Lds::swz_v(row);
        dl_k[n] = (uint32_t)row * kv_pitch * 2u + (uint32_t)(16 * sk);
        dl_v[n] = (uint32_t)row * kv_pitch * 2u + (uint32_t)(16 * sv);
        dl_k_on[n] = __ballot(8 * sk < D);
        dl_v_on[n] = __ballot(8 * sv < D);
        if (n >= Lds::SETS) {  // (the same columns, rows on: known to the compiler)
            dl_k[n] = dl_k[n % Lds::SETS] + (uint32_t)Lds::rows_on(n) * kv_pitch * 2u;
            dl_v[n] = dl_v[n % Lds::SETS] + (uint32_t)Lds::rows_on(n) * kv_pitch * 2u;
            dl_k_on[n] = dl_k_on[n % Lds::SETS];
            dl_v_on[n] = dl_v_on[n % Lds::SETS];
        }
    }
    if constexpr (DIRECT && !WHOLE) {
#pragma unroll
        for (int n = 0; n < NLD; n++) {
            unsigned char* const at = lds + half_at + Lds::block(wave, n) + 16 * lane;
#pragma unroll
            for (int st = 0; st < Lds::CLEARED; st++)
                if (!(((st < 2 ? dl_k_on : dl_v_on)[n] >> lane) & 1)) *(u32x4_t*)(at + st * STAGE_B) = u32x4_t{0u, 0u, 0u, 0u};
        }
    }
    // the tile whose first row lies tile_off bytes into the descriptor -> the stage at stage_off
    auto dl_tile = [&](const u32x4_t& rs, const uint32_t (&lane_off)[NLD], const uint64_t (&on)[NLD], uint32_t tile_off, uint32_t stage_off) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NLD; n++) {
            const uint32_t block = lds_base + half_at + stage_off + (uint32_t)Lds::block(wave, n);
            const uint32_t lane_at = lane_off[n % Lds::SETS];
            const uint32_t off = tile_off + (uint32_t)Lds::rows_on(n) * kv_pitch * 2u;
            if constexpr (WHOLE) buffer_to_lds(rs, lane_at, off, block);
            else buffer_to_lds_of(on[n % Lds::SETS], rs, lane_at, off, block);
        }
    };
    // Tile 0 (K and V) and K of tile 1 are requested before the sequence lengths have arrived (a dependent load
    // away), through descriptors that end with the tensor's last row: the rows of V(0) past the last key are zeroed
    // once the length is known, those of K are masked in the score tile whatever they hold.  (A span of the keys
    // starts where the sequence's own length puts it: its requests wait for the lengths.)
    const uint32_t tile_bytes_g = (uint32_t)KT * kv_pitch * 2u;  // from a tile's first row to the next tile's, in memory
    if (!SPLIT && !WIN && !HALVES) {
        const uint32_t all_bytes = p.seq_kv > 0 ? ((uint32_t)(p.seq_kv - 1) * kv_pitch + (uint32_t)D) * 2u : 0u;
        if constexpr (DIRECT) {
            const u32x4_t Kall = make_rsrc(Kg, all_bytes), Vall = make_rsrc(Vg, all_bytes);
            dl_tile(Kall, dl_k, dl_k_on, 0u, 0u);
            dl_tile(Vall, dl_v, dl_v_on, 0u, 2u * STAGE_B);
            dl_tile(Kall, dl_k, dl_k_on, tile_bytes_g, STAGE_B);
        } else {
            const __amdgpu_buffer_rsrc_t Kall = __builtin_amdgcn_make_buffer_rsrc((void*)Kg, 0, all_bytes, kBufferFlags);
            const __amdgpu_buffer_rsrc_t Vall = __builtin_amdgcn_make_buffer_rsrc((void*)Vg, 0, all_bytes, kBufferFlags);
#pragma unroll
            for (int n = 0; n < NL; n++) {
                kreg[0][n] = __builtin_amdgcn_raw_buffer_load_b128(Kall, ld_off[n], 0, 0);
                vreg[0][n] = __builtin_amdgcn_raw_buffer_load_b128(Vall, ld_off[n], 0, 0);
                k1[n] = PIPE ? __builtin_amdgcn_raw_buffer_load_b128(Kall, ld_off[n], tile_bytes_g, 0) : u32x4_t{0u, 0u, 0u, 0u};
            }
        }
    }

    // The rest of the arguments, requested together: left to itself the compiler loads a field where it is first used
    // and waits for a line at a time.
    if constexpr (MODE == kMaskPadding) asm volatile("" ::"s"(p.keep), "s"(p.ref_bc));
    asm volatile("" ::"s"(p.q), "s"(p.out), "s"(p.q_lens), "s"(p.kv_lens), "s"(p.seq_q), "s"(p.zero_padded_rows), "s"(p.scale_log2e),
                 "s"(p.lq.batch_stride), "s"(p.lq.head_stride), "s"(p.lq.row_pitch), "s"(p.lo.batch_stride),
                 "s"(p.lo.head_stride), "s"(p.lo.row_pitch));

    // (The lengths are read through the constant address space -- nothing writes them during the launch: behind assembly
    // statements, which count as writers of memory, the compiler would otherwise fetch them with vector loads, and a wait
    // for a vector load is a wait for every request issued before it: 30.7 us instead of 29.9 on a padded batch of 16 x 16
    // heads of up to 1024 rows, 20.3 instead of 18.8 on one of 22 x 16 heads of up to 300 at head dim 80)
    auto len_at = [](const int32_t* a, int i) __attribute__((always_inline)) {
        return ((const __attribute__((address_space(4))) int32_t*)(uintptr_t)a)[i];
    };
    const int q_len_raw = p.q_lens ? (kByLength && place.b >= 0 ? place.len : len_at(p.q_lens, b)) : p.seq_q;
    // (a padded batch of self-attention hands over one array for both: one dependent load instead of two in a row)
    const int kv_len_raw = p.kv_lens ? (p.kv_lens == p.q_lens ? q_len_raw : len_at(p.kv_lens, b)) : p.seq_kv;
    const int n_q = min(max(q_len_raw, 0), p.seq_q);  // valid query positions
    int n_keys = min(max(kv_len_raw, 0), p.seq_kv);  // keys that exist
    int qtile = SPLIT ? zz / p.n_splits : zz;
    const int split = SPLIT ? zz - qtile * p.n_splits : 0;
    (void)split;
    // A padded batch ranks each sequence's OWN query tiles, last (longest) first: rank 0 is the tile that holds the
    // sequence's last valid row, and the tiles of padded rows only, which have nothing to walk, take the ranks behind
    // the valid ones and so are dispatched last, into the gaps at the end, instead of holding the first slots.
    if (!SPLIT && p.q_lens) {
        const int n_qt = (n_q * G + TROWS - 1) / TROWS;  // tiles with valid rows
        const int rank = (int)blockIdx.z;
        qtile = rank < n_qt ? n_qt - 1 - rank : rank;
        if (kByLength && place.b >= 0) qtile = place.qtile;
    }
    const int q0 = qtile * TROWS;
    // which 32 query rows of the tile a wave owns.  Wave w runs on SIMD w % 4, and under a causal mask the rows at
    // the end of a tile see more keys than those at its start: the assignment rotates from workgroup to workgroup
    // so that no SIMD collects the long rows of every tile.
    const int wq = (wave + hx + b + (int)blockIdx.z) & 3;
    int off = n_keys - n_q;  // causal: the last valid query sees every key

    // keys the workgroup walks
    int kv_end = n_keys;
    {
        const int s_first = G > 1 ? q0 / G : q0;
        const int s_last = min(G > 1 ? (q0 + TROWS - 1) / G : (q0 + TROWS - 1), n_q - 1);
        if (kCausal) kv_end = min(n_keys, s_last + off + 1);
        if (s_first >= n_q) kv_end = 0;  // a tile of padded query rows only
        kv_end = max(kv_end, 0);
    }
    int n_tiles = (kv_end + KT - 1) / KT;
    if (SPLIT) {
        // this workgroup's span of the walk: tiles [t_begin, t_end).  From here on keys are counted from the span's
        // first key: the tensors' base, the key count, the causal offset and the end of the walk all move by it, and
        // the walk below is that of a sequence whose keys are the span's (a row whose last visible key lies before the
        // span gets a negative limit: every score masked, an empty partial).
        const int per = (n_tiles + p.n_splits - 1) / p.n_splits;
        const int t_begin = split * per, t_end = min(n_tiles, t_begin + per);
        const int key0 = t_begin * KT;
        n_tiles = max(t_end - t_begin, 0);
        kv_end = min(kv_end, t_end * KT) - key0;
        n_keys = min(n_keys, t_end * KT) - key0;
        off -= key0;
        Kg += (size_t)key0 * (size_t)p.lkv.row_pitch;
        Vg += (size_t)key0 * (size_t)p.lkv.row_pitch;
    }
    if (WIN) {
        // the first key any row of the workgroup sees, rounded down to a tile: the walk starts there
        const int key0 = (max(q0 + off - p.window + 1, 0) / KT) * KT;
        n_tiles = max(n_tiles - key0 / KT, 0);
        kv_end -= key0;
        n_keys -= key0;
        off -= key0;
        Kg += (size_t)key0 * (size_t)p.lkv.row_pitch;
        Vg += (size_t)key0 * (size_t)p.lkv.row_pitch;
    }
    const int n_loop = HALVES ? (n_tiles + 1) / 2 : n_tiles;  // tiles between the workgroup's barriers
    int half_key0 = 0;
    if (HALVES) {  // this half's span of the walk, as a span of SPLIT; the second may be a tile shorter
        half_key0 = half * n_loop * KT;
        n_tiles = half ? n_tiles - n_loop : n_loop;
        n_keys = min(n_keys, (half + 1) * n_loop * KT) - half_key0;
        off -= half_key0;
        Kg += (size_t)half_key0 * (size_t)p.lkv.row_pitch;
        Vg += (size_t)half_key0 * (size_t)p.lkv.row_pitch;
    }
    auto store_row = [&](uint16_t* dst, u32x4_t v) __attribute__((always_inline)) {  // PAST: past the caches (out_goes_past)
        if constexpr (PAST) store_past(dst, v);
        else *(u32x4_t*)dst = v;
    };
    // A tile of padded query rows only (a padded batch has many: every tile behind a sequence's last row) has nothing
    // to load or walk: its rows get the fill value and the workgroup is done.
    if (!SPLIT && !PACKED && q0 >= n_q) {
        const uint32_t f2 = p.zero_padded_rows ? 0u : 0x7fc07fc0u;
        const u32x4_t val = {f2, f2, f2, f2};
        uint16_t* const ob = p.out + (size_t)b * p.lo.batch_stride + (size_t)h0 * p.lo.head_stride;
        if (HALVES && half) return;
        for (int c = tid; c < TROWS * CH; c += TTHREADS) {
            const int row = c / CH, ch = c - row * CH;
            if (q0 + row < rows_total && 8 * ch < D) store_row(ob + (size_t)(q0 + row) * p.lo.row_pitch + 8 * ch, val);
        }
        // (the early requests land in this workgroup's LDS: not to be left in flight when it is handed on)
        if constexpr (DIRECT) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }
    // K and V are read through buffer descriptors that end with the last key's row: a request for a row behind it
    // returns zeros without touching memory.  Zero rows of V are what the walk needs there (their weights are zero,
    // and zero times a copy of a non-finite row would be NaN); zero rows of K give score 0, masked like any score
    // past the last key.  The lane's offset is a constant of the thread and the tile's offset a scalar, so a request
    // costs no address arithmetic.  (Offsets are 32-bit: the launcher refuses slabs of 4 GiB and more.)
    const uint32_t slab_bytes = n_keys > 0 ? ((uint32_t)(n_keys - 1) * kv_pitch + (uint32_t)D) * 2u : 0u;
    const __amdgpu_buffer_rsrc_t Kbuf = __builtin_amdgcn_make_buffer_rsrc((void*)Kg, 0, slab_bytes, kBufferFlags);
    const __amdgpu_buffer_rsrc_t Vbuf = __builtin_amdgcn_make_buffer_rsrc((void*)Vg, 0, slab_bytes, kBufferFlags);
    const u32x4_t Kd = make_rsrc(Kg, slab_bytes), Vd = make_rsrc(Vg, slab_bytes);  // (DIRECT: the same descriptors as scalars)
    if (DIRECT && (SPLIT || WIN || HALVES)) {
        dl_tile(Kd, dl_k, dl_k_on, 0u, 0u);
        dl_tile(Vd, dl_v, dl_v_on, 0u, 2u * STAGE_B);
        dl_tile(Kd, dl_k, dl_k_on, tile_bytes_g, STAGE_B);
    } else if (SPLIT || WIN) {  // tile 0 (K and V) and K of tile 1 of the span / of the window
#pragma unroll
        for (int n = 0; n < NL; n++) {
            kreg[0][n] = __builtin_amdgcn_raw_buffer_load_b128(Kbuf, ld_off[n], 0, 0);
            vreg[0][n] = __builtin_amdgcn_raw_buffer_load_b128(Vbuf, ld_off[n], 0, 0);
            k1[n] = PIPE ? __builtin_amdgcn_raw_buffer_load_b128(Kbuf, ld_off[n], tile_bytes_g, 0) : u32x4_t{0u, 0u, 0u, 0u};
        }
    } else if (!DIRECT && n_keys < KT) {  // the early requests ended with the tensor, not with the sequence
#pragma unroll
        for (int n = 0; n < NL; n++)
            if ((tid + TTHREADS * n) / CH >= n_keys) vreg[0][n] = u32x4_t{0u, 0u, 0u, 0u};
    }

    if (MODE == kMaskPadding && !DIRECT && n_keys > 0) {  // keep bytes past the last key count as kept: `lim` masks those keys
        const int j = lane & (KT - 1);
        const uint32_t kb = p.keep[min(j, n_keys - 1)];
        keep_raw[0] = j < n_keys ? kb : 1u;
    }

    f32x16_t acc_o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc_o[t][i] = 0.0f;
    float m_run = neg_inf(), l_run = 0.0f;
    bool poison = false;
    bool valid = false;
    const float cc = BIAS ? kLog2e : p.scale_log2e;  // exp2 argument per unit of score

    if (n_loop > 0) {
        static_assert(CHUNKS % TTHREADS == 0, "every thread moves NL chunks of every tile");
        // Every request below is unconditional -- a tile index past the last tile is clamped to it, a chunk past the
        // head dim reads column 0 -- and only the LDS write is predicated.  With no branch around a load the compiler
        // counts the loads in flight exactly and waits at a park for the oldest register set only; with one it
        // falls back to waiting for all of them, which empties the prefetch queue at every tile.
        if (!DIRECT && D < DP) {  // the columns that are never parked are zero in both stages
            for (int i = tid; i < Cfg::TILE_BYTES / 16; i += TTHREADS) ((u32x4_t*)lds)[i] = u32x4_t{0u, 0u, 0u, 0u};
            __syncthreads();
        }
        const int last_kv0 = (n_tiles - 1) * KT;
        auto issue_k = [&](u32x4_t (&dst)[NL], int kv0) __attribute__((always_inline)) {
            const uint32_t tile_off = (uint32_t)min(kv0, last_kv0) * (kv_pitch * 2u);
#pragma unroll
            for (int n = 0; n < NL; n++) dst[n] = __builtin_amdgcn_raw_buffer_load_b128(Kbuf, ld_off[n], tile_off, 0);
        };
        auto issue_v = [&](auto set_c, int kv0) __attribute__((always_inline)) {
            constexpr int SET = decltype(set_c)::value;
            kv0 = min(kv0, last_kv0);
            const uint32_t tile_off = (uint32_t)kv0 * (kv_pitch * 2u);
#pragma unroll
            for (int n = 0; n < NL; n++) vreg[SET][n] = __builtin_amdgcn_raw_buffer_load_b128(Vbuf, ld_off[n], tile_off, 0);
            // key-padding vector of the tile: one byte per lane, turned into bits with a ballot when the tile is parked
            if (MODE == kMaskPadding) {
                const int j = kv0 + (lane & (KT - 1));
                const uint32_t kb = p.keep[min(j, n_keys - 1)];
                keep_raw[SET] = (j < n_keys) ? kb : 1u;  // keys past the end are masked by `lim`
            }
        };
        auto park_k = [&](const u32x4_t (&src)[NL], int st) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NL; n++)
                if (D == DP || ld_on[n]) *(u32x4_t*)(lds + st * (KT * LDK * 2) + st_k[n]) = src[n];
        };
        // Mask::Padding, DIRECT: a bit per key in LDS, behind V(1)'s stage, where half of the query rows came in; a wave reads
        // the word of its next item a step ahead
        constexpr bool KEEP_BITS = MODE == kMaskPadding && DIRECT;
        static_assert(!KEEP_BITS || QLDS, "the bits take the query rows' place");
        constexpr int kKeepAt = Lds::KEEP_AT;
        uint32_t keep_word_next = ~0u;
        uint64_t keep_cur = ~0ull, keep_next = ~0ull;  // keep bits of the tile whose items are in their softmax step, and of the next
        auto park_v = [&](auto set_c, int st) __attribute__((always_inline)) {
            constexpr int SET = decltype(set_c)::value;
#pragma unroll
            for (int n = 0; n < NL; n++)
                if (D == DP || ld_on[n]) *(u32x4_t*)(lds + st * (KT * LDV * 2) + st_v[n]) = vreg[SET][n];
            if (MODE == kMaskPadding) keep_next = __ballot(keep_raw[SET] != 0);
        };

        // ---- this lane's query row
        const int r = q0 + 32 * wq + col;
        const int s_pos = G > 1 ? r / G : r;
        const bool exists = r < rows_total;
        valid = exists && s_pos < n_q;
        int lim = n_keys - 1;  // last key this row sees
        if (kCausal) lim = min(lim, s_pos + off);
        if (!valid) lim = -1;
        // the largest and smallest `lim` of the wave, as scalars (the tests on them are wave-uniform): lim grows with
        // the row, and the rows that are not valid are the last ones
        int wave_lim_max, wave_lim_min;
        {
            const int r_first = q0 + 32 * wq, r_last = r_first + 31;
            const int r_lim = min(rows_total, n_q * G);  // rows below it are valid
            const int r_top = min(r_last, r_lim - 1);
            const int s_top = G > 1 ? r_top / G : r_top, s_bot = G > 1 ? r_first / G : r_first;
            wave_lim_max = r_first < r_lim ? (kCausal ? min(n_keys - 1, s_top + off) : n_keys - 1) : -1;
            wave_lim_min = r_last < r_lim ? (kCausal ? min(n_keys - 1, s_bot + off) : n_keys - 1) : -1;
        }
        // items this wave walks: the ones that hold a key some row of it sees (a prefix of the workgroup's items)
        const int n_it = wave_lim_max < 0 ? 0 : min(n_tiles * NI, (wave_lim_max >> 5) + 1);
        // a window: the first key this row sees, and the largest such key over the wave's rows (its last valid row's)
        const int lo = WIN ? max(lim - p.window + 1, 0) : 0;
        const int wave_lo_max = WIN ? max(wave_lim_max - p.window + 1, 0) : 0;

        // (the query row is read without a test: a row past the tensor reads the tensor's last row)
        const int r_q = min(r, rows_total - 1);
        const int s_q = G > 1 ? r_q / G : r_q;
        const size_t q_off = (size_t)b * p.lq.batch_stride + (size_t)(h0 + (r_q - s_q * G)) * p.lq.head_stride + (size_t)s_q * p.lq.row_pitch;

        // BIAS (scores = (q . k) * scale + bias, crates/rustorch-nn/src/attention.rs:378-392, kept in the natural domain so
        // that a bias of -1e4 weighs as it does in the reference): f32 rows of seq_kv per (batch, head), or one matrix for
        // all.  An item's 32 rows of 32 keys go from memory to the wave's own 4 KB of LDS as whole 128-byte pieces of a row
        // (8 rows a load instruction), and from there into the order the scores
        // sit in; the 16-byte slots of a row are XORed with bits of the row, as those of a K tile of 128-byte rows.  Read
        // from its row in memory by each lane, 16 bytes of 32 rows at a time, the bias kept the address unit busy for half
        // of the launch and the waves waiting for 54 % of theirs: B=4 H=16 T=1024 hd=64 47.4 -> 28.3 us with warm inputs and
        // 47.3 -> 29.9 with inputs that change from pass to pass.  Keys behind the last one read the next row, or zeros behind the tensor:
        // those scores are masked.
        // A row may start at any multiple of 4 bytes: a 16-byte request asks for no more of its address.  The one chunk that must
        // not be asked for whole is that which ends behind the tensor: the wave of the tensor's last row takes an item that is short
        // of 32 keys 4 bytes a lane, 2 rows an instruction.  us, every request for an unaligned tensor that way -> now, B H T head dim,
        // one matrix for all: 4 16 1023 64 36.8 -> 33.0 (1024 keys 30.2), 13 12 1662 32 190 -> 182 (1664 144), 4 12 1662 128 113 -> 103, 1 12
        // 161 32 7.9 -> 7.1, 4 8 1023 256 62.8 -> 58.9; one a head: 2 8 466 80 17.3 -> 15.5, 1 8 77 x 513 64 14.3 -> 12.5.
        u32x4_t bias_rsrc = {0u, 0u, 0u, 0u};
        uint32_t bias_lane[2] = {0u, 0u}, bias_at = 0, bias_step = 0;
        const uint32_t bias_lds = BIAS ? (uint32_t)(kBiasAt + (wave + 4 * half) * Cfg::BIAS_BYTES) : 0u;
        int bias_whole = 0;      // items before it are asked for 16 bytes a lane
        if constexpr (BIAS) {
            const int r_first = q0 + 32 * wq, n_rows = max(min(32, rows_total - r_first), 0);
            const float* const bb = p.bias + ((size_t)b * p.heads + h0) * (size_t)p.bias_bh_stride + (size_t)min(r_first, rows_total - 1) * (size_t)p.seq_kv;
            const uint32_t pitch = (uint32_t)p.seq_kv * 4u, first = 4u * (uint32_t)min(half_key0, p.seq_kv);
            const bool ends = !p.bias_vec4 && r_first + n_rows == rows_total && (p.bias_bh_stride == 0 || (b == (int)gridDim.y - 1 && h0 == p.heads - 1));
            bias_whole = ends ? (p.seq_kv - half_key0) >> 5 : 0x7fffffff;
            bias_rsrc = make_rsrc((const char*)bb + first, n_rows > 0 ? (uint32_t)n_rows * pitch - first + (ends || p.bias_vec4 ? 0u : min(12u, pitch)) : 0u);
            // instruction n: rows 8 n + lane / 8
            const int row = lane >> 3, slot = (lane & 7) ^ (row >> 1);
            bias_lane[0] = (uint32_t)row * pitch + 16u * (uint32_t)slot;
            bias_lane[1] = (uint32_t)row * pitch + 16u * (uint32_t)(slot ^ 4);
            bias_step = 8u * pitch;
            bias_at = bias_lds + (uint32_t)(col * 128 + ((hh ^ ((col >> 1) & 7)) * 16));
        }
        auto bias_request = [&](int item) __attribute__((always_inline)) {
            const uint32_t k_off = 128u * (uint32_t)item;
            if (__builtin_expect(item < bias_whole, 1)) {
#pragma unroll
                for (int n = 0; n < 4; n++)
                    buffer_to_lds(bias_rsrc, bias_lane[n & 1], k_off + (uint32_t)n * bias_step, lds_base + bias_lds + 1024u * (uint32_t)n);
            } else {  // instruction n: rows 2 n + lane / 32
                const uint32_t pitch = (uint32_t)p.seq_kv * 4u;
#pragma unroll
                for (int n = 0; n < 16; n++)
                    buffer_to_lds_b32(bias_rsrc, (uint32_t)(lane >> 5) * pitch + ((4u * (uint32_t)(lane & 31)) ^ (16u * (uint32_t)(n & 7))), k_off + (uint32_t)(2 * n) * pitch,
                                      lds_base + bias_lds + 256u * (uint32_t)n);
            }
        };
        auto bias_read = [&](f32x4_t (&bv)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 4; j++) bv[j] = *(const f32x4_t*)(lds + (bias_at ^ (uint32_t)(32 * j)));
        };
        if constexpr (BIAS) bias_request(0);

        // Mask::Padding hiding the reference's whole first key tile: every row NaN (the tiled recurrence of
        // cpu_forward.rs:268-425 takes exp(-inf - (-inf)) on that tile and never recovers)
        const int lead = p.ref_bc < n_keys ? p.ref_bc : n_keys;
        if (MODE == kMaskPadding && !KEEP_BITS) {
            bool any = false;
            for (int j = lane; j < lead; j += kWave) any |= (p.keep[j] != 0);
            poison = !__any(any);
        }

        // ---- Q as B operand: column q = lane % 32, contraction slots 16 ks + 8 hh .. + 8
        bf16x8_t qreg[KS];
        if constexpr (QLDS) {
            // instruction n: chunks 64 n .. + 63 of the wave's 32 rows, swizzled as those of a K tile (zeros behind the last row
            // and behind the head dim)
            const int r_first = q0 + 32 * wq, n_rows = max(min(32, rows_total - r_first), 0);
            const uint32_t q_pitch = (uint32_t)p.lq.row_pitch;
            const bool many = WIN && (uint64_t)gridDim.x * gridDim.y * gridDim.z > (uint64_t)p.n_cus * Cfg::OCC_DIRECT;
            const u32x4_t Qd = make_rsrc(p.q + (size_t)b * p.lq.batch_stride + (size_t)h0 * p.lq.head_stride + (size_t)min(r_first, rows_total - 1) * q_pitch,
                                         n_rows > 0 ? ((uint32_t)(n_rows - 1) * q_pitch + (uint32_t)D) * 2u : 0u);
#pragma unroll
            for (int n = 0; n < Lds::Q_REQUESTS; n++) {
                const int c = 64 * n + lane, row = (int)((uint32_t)c / CH), slot = (c - row * CH) ^ Lds::swz_k(row);
                const uint32_t at = 8 * slot < D ? (uint32_t)row * q_pitch * 2u + 16u * (uint32_t)slot : 0x7fffffffu;
                const uint32_t block = lds_base + half_at + (uint32_t)Lds::q_block(wave, n);
                if (WIN && DP <= 64 && many) buffer_to_lds_past(Qd, at, 0u, block);
                else buffer_to_lds(Qd, at, 0u, block);
            }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if constexpr (QLDS) break;
            // Unconditional loads (a row past the tensor is read from the tensor's last row, a chunk past the head dim
            // from its last chunk): a load under a per-lane test costs a branch of its own.  A row that does not exist
            // has every score masked and is not written, so what it holds does not matter; the columns past the head
            // dim must be zero.
            const int d0 = 16 * ks + 8 * hh;
            u32x4_t z = {0u, 0u, 0u, 0u};
            if constexpr (DP <= 128 || DIRECT) {
                z = *(const u32x4_t*)(p.q + q_off + min(d0, D - 8));
                if (D < DP && d0 >= D) z = u32x4_t{0u, 0u, 0u, 0u};
            } else {  // (head dim 256 has no register to spare for the clamped addresses)
                if (exists && d0 < D) z = *(const u32x4_t*)(p.q + q_off + d0);
            }
            qreg[ks] = __builtin_bit_cast(bf16x8_t, z);
        }

        // per-lane LDS offsets (elements): K operand row `col`, slots 8 hh; V operand row (j >> 2) + 4 hh, columns 16 g16 + 4 (j & 3)
        const int k_off = col * LDK + 8 * hh;
        const int v_off = (((lane & 15) >> 2) + 4 * hh) * LDV + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        // DIRECT (byte offsets): the same operand rows and columns in the swizzled layout.  The swizzles only permute
        // address bits that the operand index also occupies, so operand ks sits at k_base ^ 32 ks, operand dt at
        // v_base ^ 64 dt; in rows of 192 bytes, whose start has bits among those, the two operands of four slots have a base
        // each, and four slots on is 64 bytes on.
        uint32_t k_base = 0, k_base1 = 0, v_base = 0;
        if constexpr (DIRECT) {
            const int j = lane & 15, g16 = (lane >> 4) & 1, vrow = (j >> 2) + 4 * hh, low = 2 * g16 + ((j & 3) >> 1);
            k_base = half_at + (uint32_t)(col * ROWB + ((hh ^ Lds::swz_k(col)) * 16));
            if constexpr (DP == 96) k_base1 = half_at + (uint32_t)(col * ROWB + (((2 + hh) ^ Lds::swz_k(col)) * 16));
            v_base = half_at + (uint32_t)(Lds::V_AT + vrow * ROWB + ((low ^ Lds::swz_v(vrow)) * 16) + 8 * (j & 1));
        }
        // where the operands of item `item` of stage `st` start: with the lane's own offset (padded layout), or without
        // it (DIRECT: load_op adds the lane's swizzled offset)
        auto k_at = [&](int st, int item) __attribute__((always_inline)) -> const uint16_t* {
            if constexpr (DIRECT) return (const uint16_t*)(lds + st * STAGE_B + item * 32 * ROWB);
            else return Ks + st * KT * LDK + item * 32 * LDK + k_off;
        };
        auto v_at = [&](int st, int item) __attribute__((always_inline)) -> const uint16_t* {
            if constexpr (DIRECT) return (const uint16_t*)(lds + st * STAGE_B + item * 32 * ROWB);
            else return Vs + st * KT * LDV + item * 32 * LDV + v_off;
        };


        constexpr int KB = 8;  // ballots of a wave whose bytes are requested together
        uint32_t keep_byte[KB];
        auto keep_load = [&](int base) __attribute__((always_inline)) {  // keys base + 256 i + 64 wave + lane
#pragma unroll
            for (int i = 0; i < KB; i++) {
                const int first = base + 256 * i + 64 * wave;
                keep_byte[i] = 1u;  // (keys past the end are masked by `lim`)
                if (first < n_keys) {
                    const uint32_t x = p.keep[min(first + lane, n_keys - 1)];
                    keep_byte[i] = first + lane < n_keys ? x : 1u;
                }
            }
        };
        if constexpr (KEEP_BITS) keep_load(0);

        // K(0), V(0) -> stage 0, K(1) -> stage 1; then the register sets take K(2) .. K(1 + PF) and V(1) .. V(PF)
        // (K(j) travels in set j % PF, and so does V(j))
        f32x4_t bv[4] = {};  // bias values of the item whose softmax step comes next
        auto bias_first = [&]() __attribute__((always_inline)) {
            if constexpr (BIAS) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                bias_read(bv);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                bias_request(1);
            }
        };
        if constexpr (DIRECT) {
            // tile 0 and K(1) have landed (and the queries); V rows of tile 0 past the last key, requested before the
            // lengths were known, are zeroed by the lane that fetched them
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if constexpr (QLDS) {
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const unsigned char* const at = lds + Lds::q_block(wave, 0);
                    qreg[ks] = *(const bf16x8_t*)(at + (DP == 96 ? ((ks & 1) ? k_base1 : k_base) + (uint32_t)(64 * (ks >> 1)) : k_base ^ (uint32_t)(32 * ks)));
                }
            }
            if (n_keys < KT) {
#pragma unroll
                for (int n = 0; n < NLD; n++)
                    if (dl_row[n] >= n_keys) *(u32x4_t*)(lds + half_at + Lds::V_AT + Lds::block(wave, n) + 16 * lane) = u32x4_t{0u, 0u, 0u, 0u};
            }
            bias_first();
            if constexpr (KEEP_BITS) {
                __syncthreads();  // every wave has read its query rows
                for (int base = 0;;) {
#pragma unroll
                    for (int i = 0; i < KB; i++) {
                        const int first = base + 256 * i + 64 * wave;
                        const uint64_t bits = __ballot(keep_byte[i] != 0);
                        if (lane == 0 && first < n_keys) *(u32x2_t*)(lds + kKeepAt + first / 8) = u32x2_t{(uint32_t)bits, (uint32_t)(bits >> 32)};
                    }
                    base += 256 * KB;
                    if (base >= n_keys) break;
                    keep_load(base);
                }
            }
        } else {
            park_k(kreg[0], 0);
            park_v(std::integral_constant<int, 0>{}, 0);
            keep_cur = keep_next;
            if (PIPE) park_k(k1, 1);
            bias_first();
            {
                auto prefetch = [&](auto i_c) __attribute__((always_inline)) {
                    constexpr int I = decltype(i_c)::value;  // 0 .. PF - 1
                    constexpr int KA = PIPE ? 2 : 1;         // K runs a tile ahead of V in the pipelined walk only
                    issue_k(kreg[(KA + I) % PF], (KA + I) * KT);
                    issue_v(std::integral_constant<int, (1 + I) % PF>{}, (1 + I) * KT);
                };
                prefetch(std::integral_constant<int, 0>{});
                if (PF >= 2) prefetch(std::integral_constant<int, 1>{});
                if (PF >= 3) prefetch(std::integral_constant<int, 2>{});
                static_assert(PF <= 3, "prologue covers up to three sets");
            }
        }
        __syncthreads();
        if constexpr (KEEP_BITS) {
            keep_word_next = *(const uint32_t*)(lds + kKeepAt);
            bool any = false;
            for (int j = lane; 32 * j < lead; j += kWave)
                any |= (*(const uint32_t*)(lds + kKeepAt + 4 * j) & (lead - 32 * j >= 32 ? ~0u : (1u << (lead - 32 * j)) - 1u)) != 0;
            poison = !__any(any);
        }

        // ---- pieces of a step
        // the bias, then the masks, on the scores of the item whose keys start at k0 (item `it` of its tile)
        auto mask_item = [&](int it, int k0, f32x16_t& sc) __attribute__((always_inline)) {
            if (BIAS) {
#pragma unroll
                for (int i = 0; i < 16; i++) sc[i] = __builtin_fmaf(sc[i], p.scale, bv[i >> 2][i & 3]);
            }
            if (k0 + 31 > wave_lim_min) {
                // key k0 + 8 (i / 4) + 4 hh + i % 4 is hidden when it lies past lim: one subtraction per item, then a
                // comparison with a constant per score
                const int room = lim - k0 - 4 * hh;
#pragma unroll
                for (int i = 0; i < 16; i++) sc[i] = (8 * (i >> 2) + (i & 3) > room) ? neg_inf() : sc[i];
            }
            if (WIN && k0 < wave_lo_max) {
                const int room_lo = lo - k0 - 4 * hh;  // key k0 + 8 (i / 4) + 4 hh + i % 4 lies before the window when below lo
#pragma unroll
                for (int i = 0; i < 16; i++) sc[i] = (8 * (i >> 2) + (i & 3) < room_lo) ? neg_inf() : sc[i];
            }
            if (MODE == kMaskPadding) {
                const uint32_t keep_word = KEEP_BITS ? (uint32_t)__builtin_amdgcn_readfirstlane(keep_word_next) : (uint32_t)(keep_cur >> (32 * it));
                if (keep_word != 0xffffffffu) {
                    const uint32_t mine = keep_word >> (4 * hh);  // bit 8(i/4) + i%4 of `mine` is key 8(i/4) + 4hh + i%4
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const bool kept = (mine >> (8 * (i >> 2) + (i & 3))) & 1u;
                        sc[i] = kept ? sc[i] : neg_inf();
                    }
                }
            }
        };
        // operand m of a step: even m = K rows of the next item (A operand of score instruction m / 2), odd m = V of
        // the previous item (contraction slots 0-3 of a lane are keys 16u + 4hh + 0..3, slots 4-7 keys 16u + 8 + 4hh + 0..3)
        auto load_op = [&](int m, const uint16_t* kp, const uint16_t* vp) __attribute__((always_inline)) {
            if constexpr (DIRECT) {
                const int i = m >> 1, u = i / DT, dt = i - u * DT;
                if ((m & 1) == 0) {
                    if constexpr (DP == 96) return *(const u32x4_t*)((const unsigned char*)kp + ((i & 1) ? k_base1 : k_base) + 64 * (i >> 1));
                    return *(const u32x4_t*)((const unsigned char*)kp + (k_base ^ (uint32_t)(32 * i)));
                }
                const unsigned char* const vq = (const unsigned char*)vp + (DP == 96 ? v_base + (uint32_t)(64 * dt) : (v_base ^ (uint32_t)(64 * dt))) + 16 * u * ROWB;
                const u32x2_t lo = t_lds_read_tr16((const uint16_t*)vq);
                const u32x2_t hi = t_lds_read_tr16((const uint16_t*)(vq + 8 * ROWB));
                return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
            }
            if ((m & 1) == 0) return *(const u32x4_t*)(kp + 16 * (m >> 1));
            const int i = m >> 1, u = i / DT, dt = i - u * DT;
            const u32x2_t lo = t_lds_read_tr16(vp + 16 * u * LDV + 32 * dt);
            const u32x2_t hi = t_lds_read_tr16(vp + 16 * u * LDV + 32 * dt + 8 * LDV);
            return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        };
        // An empty assembly statement that takes x as a read-write argument: whatever makes x stays above it, whatever
        // uses x stays below.  A run of them is a fence for exactly the values named.
        auto pin_f = [](float& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
        auto pin_u = [](uint32_t& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
        auto pin_b = [](bf16x8_t& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };

        float neg_mc = valid ? __uint_as_float(0x7f800000u) : 0.0f;  // -m_run * cc; +inf while a valid row has no max yet
        // The values that travel from step to step come in pairs: a step reads one of a pair and writes the other, and
        // the next step has them the other way round, so nothing is copied.
        f32x16_t s_a, s_b;        // S(j), made in step j - 1, and S(j + 1)
        bf16x8_t p_a[2], p_b[2];  // P(j - 1) and P(j)
        p_a[0] = p_a[1] = p_b[0] = p_b[1] = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});

        // A window: the items ahead of the first that a row of the wave sees are left out (1.5 of 10.5 items a wave at 256
        // keys, 1.5 and more of 4.5 at 64, each on the slow path of rows without a maximum); the wave only keeps its part of
        // the movement.
        const int j_first = WIN && n_it > 0 ? max(min(n_keys - 1, q0 + 32 * wq + off) - p.window + 1, 0) >> 5 : 0;
        // Its last rows' first key lies in the item behind, but for a window of 1 mod 32: they get their running max from that
        // item's scores, once the first step has made them (late_max, on every way into the walk: a row without a maximum
        // weighs its keys by exp2 of the plain scores).  Without a max the wave took the slow path twice.  Both together, us
        // with inputs that change from pass to pass, B H N hd window: 4 16 4096 64 256 49.2 -> 47.8, 2 16 2048 64 300 17.7 ->
        // 17.1, 1 32 1000 128 64 11.7 -> 10.6, 2 32 3000 32 500 34.7 -> 33.4, 1 8 16000 128 2500 165.2 -> 160.9, 3 12 3001 80
        // 77 30.1 -> 27.8, 4 28 1900 96 150 49.1 -> 45.4.
        const bool late = WIN && PIPE && n_it > j_first + 1 && wave_lo_max > 32 * j_first + 31;

        // S of the wave's first item (0, or under a window the first that a row of it sees), before its pipeline starts
#pragma unroll
        for (int i = 0; i < 16; i++) s_a[i] = s_b[i] = 0.0f;
        auto first_scores = [&](int it, int k0, const uint16_t* kp, f32x16_t& s) __attribute__((always_inline)) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, load_op(2 * ks, kp, nullptr)), qreg[ks], s, 0, 0, 0);
            // The running max starts at the max of this item, taken here, so that the first step already runs the
            // fast path (without it the step would form P twice and rescale an O that is still zero).  A bias goes on a
            // copy: the step applies it to the scores.  (Masks applied twice change nothing.)
            f32x16_t s_0;
            if (BIAS) s_0 = s;
            mask_item(it, k0, BIAS ? s_0 : s);
            const float m0 = t_max_with_other_half(t_max16(BIAS ? s_0 : s));
            if (m0 > neg_inf()) {  // (false for -inf and for NaN: such a row waits for the slow path)
                m_run = m0;
                neg_mc = -m0 * cc;
            } else if (late) {
                neg_mc = 0.0f;  // every score of the row is masked, and weighs exp2(-inf + 0)
            }
        };
        auto late_max = [&](int it, int k0, f32x16_t& s) __attribute__((always_inline)) {
            if (!late) return;
            mask_item(it, k0, s);
            const float m1 = t_max_with_other_half(t_max16(s));
            if (m_run == neg_inf()) {
                m_run = m1;
                neg_mc = (m1 == neg_inf()) ? (valid ? __uint_as_float(0x7f800000u) : 0.0f) : -m1 * cc;
            }
        };
        if (PIPE && !WIN && n_it > 0) first_scores(0, 0, k_at(0, 0), s_a);

        // O^T += V(j-1)^T . P(j-1)^T alone: behind the wave's last item
        auto drain = [&](const uint16_t* vp) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const int u = i / DT, dt = i - u * DT;
                const u32x4_t av = load_op(2 * i + 1, nullptr, vp);
                acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, av), p_a[u], acc_o[dt], 0, 0, 0);
            }
        };
        // P = exp2(s * cc + nmc) of the 16 scores a lane holds as the item's two B operands, and the lane's share of
        // the row sum (plain additions: v_dot2c_f32_bf16 would halve their number but runs on the matrix pipe, where
        // it queues behind the matrix instructions of every wave of the SIMD)
        auto exp_plain = [&](const f32x16_t& sc, float nmc, uint32_t (&w)[8], float& part) __attribute__((always_inline)) {
            float part0 = 0.0f, part1 = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * e], cc, nmc));
                const float x1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * e + 1], cc, nmc));
                part0 += x0;
                part1 += x1;
                w[e] = t_cvt_pk_bf16(x0, x1);
            }
            part = part0 + part1;
        };

        // the slow path of a softmax step: the item max, O and l rescaled to it, P again from the scores
        auto raise_max_and_redo = [&](const f32x16_t& sc, uint32_t (&w)[8], float& part) __attribute__((always_inline)) {
            const float m_item = t_max_with_other_half(t_max16(sc));
            const float m_new = t_vmax(m_run, m_item);
            const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * cc);  // m_run = -inf -> 0
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int tt = 0; tt < DT; tt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc_o[tt][i] *= alpha;
            const float mc = m_use * cc;
            // a valid row that has seen no key yet keeps taking this path (and gets P = 0 from it: exp2(-inf - 0))
            neg_mc = (m_new == neg_inf()) ? (valid ? __uint_as_float(0x7f800000u) : 0.0f) : -mc;
            exp_plain(sc, -mc, w, part);
        };
        // BIAS: the next item's bias values leave LDS at the end of a step, and the values of the item behind it are
        // requested over them.  WAIT: requests made since that may still be on their way.
        auto bias_take = [&](auto wait_c) __attribute__((always_inline)) {
            if constexpr (BIAS) {
                constexpr int WAIT = decltype(wait_c)::value;
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT) : "memory");
                bias_read(bv);
            }
        };
        auto bias_ahead = [&](int k0) __attribute__((always_inline)) {
            if constexpr (BIAS) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                bias_request((k0 >> 5) + 2);
            }
        };
        // An item whose three phases run one after the other (head dims above 128): S, the softmax step, P.V
        auto step_simple = [&](int it, int k0, const uint16_t* kp, const uint16_t* vp) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 16; i++) s_a[i] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                s_a = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8_t*)(kp + 16 * ks), qreg[ks], s_a, 0, 0, 0);
            mask_item(it, k0, s_a);
            bias_take(std::integral_constant<int, 0>{});
            uint32_t w[8];
            float part;
            exp_plain(s_a, neg_mc, w, part);
            if (__builtin_expect(__any(!(part <= kTileTrigSum)), 0)) raise_max_and_redo(s_a, w, part);
            l_run += part;
            p_a[0] = __builtin_bit_cast(bf16x8_t, u32x4_t{w[0], w[1], w[2], w[3]});
            p_a[1] = __builtin_bit_cast(bf16x8_t, u32x4_t{w[4], w[5], w[6], w[7]});
            bias_ahead(k0);
            drain(vp);
        };

        // One step of the pipeline: item j (keys k0 .., item `it` of its tile) gets its softmax step; K rows of item
        // j + 1 are at kp, V rows of item j - 1 at vp.
        //
        // The softmax step takes no row max in the steady state: P is formed against the running max as it stands (a
        // stale max scales a row's P, O and l by one common factor, harmless until it overflows), and the lane's share
        // of the row sum, which is needed anyway, bounds every P of the lane.  Only when a share passes kTileTrigSum, or
        // is not a number, or a valid row has no max yet (neg_mc = +inf), does the wave take the item max, rescale O and
        // l and form P again from the scores, which are still in their registers.
        //
        // The vector work is laid out in six groups (arguments, exponentials, sums and conversions, for either half of
        // the scores), the step's matrix instructions are dealt to the groups in order, S and P.V alternating (a chain
        // on one accumulator waits for itself), and an operand is read from LDS one or two groups ahead of its instruction.
        // The fences between the groups name the vector values and the B operands of the matrix instructions on
        // either side, which is what keeps each matrix instruction inside its group.
        auto step = [&](int it, int k0, const uint16_t* kp, const uint16_t* vp, f32x16_t& s_cur, f32x16_t& s_next,
                        bf16x8_t (&p_prev)[2], bf16x8_t (&p_new)[2], auto wait_c) __attribute__((always_inline)) {
            mask_item(it, k0, s_cur);
            if constexpr (KEEP_BITS) keep_word_next = *(const uint32_t*)(lds + kKeepAt + min((k0 >> 5) + 1, (n_keys - 1) >> 5) * 4);
#pragma unroll
            for (int i = 0; i < 16; i++) s_next[i] = 0.0f;
            u32x4_t ops[NM];
            auto group_of = [](int m) __attribute__((always_inline)) { return NM >= 6 ? m * 6 / NM : (m * 6 + NM - 1) / NM; };
            auto fetch_group = [&](int gq) __attribute__((always_inline)) {
#pragma unroll
                for (int m = 0; m < NM; m++)
                    if (group_of(m) == gq) ops[m] = load_op(m, kp, vp);
            };
            auto fence_b = [&](int gq) __attribute__((always_inline)) {  // the B operands of the matrix instructions of group gq
#pragma unroll
                for (int m = 0; m < NM; m++) {
                    if (group_of(m) != gq) continue;
                    if (m & 1) pin_b(p_prev[(m >> 1) / DT]);
                    else pin_b(qreg[m >> 1]);
                }
            };
            auto multiply_group = [&](int gq) __attribute__((always_inline)) {
#pragma unroll
                for (int m = 0; m < NM; m++) {
                    if (group_of(m) != gq) continue;
                    const bf16x8_t a_op = __builtin_bit_cast(bf16x8_t, ops[m]);
                    if ((m & 1) == 0) {
                        s_next = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_op, qreg[m >> 1], s_next, 0, 0, 0);
                    } else {
                        const int i = m >> 1, u = i / DT, dt = i - u * DT;
                        acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_op, p_prev[u], acc_o[dt], 0, 0, 0);
                    }
                }
            };
            float t[8];
            uint32_t w[8];
            float part0 = 0.0f, part1 = 0.0f;
            constexpr int LOOK = DP <= 64 ? 2 : 1;  // groups between an operand's LDS read and its matrix instruction
            fetch_group(0);
            if (LOOK > 1) fetch_group(1);
            fence_b(0);
#pragma unroll
            for (int gq = 0; gq < 6; gq++) {
                if (gq + LOOK < 6) fetch_group(gq + LOOK);
                if (gq == 4) bias_take(wait_c);
                multiply_group(gq);
                const int half = gq / 3;
                if (gq % 3 == 0) {
#pragma unroll
                    for (int i = 0; i < 8; i++) t[i] = __builtin_fmaf(s_cur[8 * half + i], cc, neg_mc);
                } else if (gq % 3 == 1) {
#pragma unroll
                    for (int i = 0; i < 8; i++) t[i] = __builtin_amdgcn_exp2f(t[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; i += 2) {
                        part0 += t[i];
                        part1 += t[i + 1];
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) w[4 * half + e] = t_cvt_pk_bf16(t[2 * e], t[2 * e + 1]);
                }
                // the fence behind group gq
#pragma unroll
                for (int i = 0; i < 8; i++) pin_f(t[i]);
                if (gq % 3 == 2) {
                    pin_f(part0);
                    pin_f(part1);
#pragma unroll
                    for (int e = 0; e < 4; e++) pin_u(w[4 * half + e]);
                }
                fence_b(gq);
                if (gq + 1 < 6) fence_b(gq + 1);
            }
            bias_ahead(k0);
            float part = part0 + part1;
            if (__builtin_expect(__any(!(part <= kTileTrigSum)), 0)) raise_max_and_redo(s_cur, w, part);
            l_run += part;
            p_new[0] = __builtin_bit_cast(bf16x8_t, u32x4_t{w[0], w[1], w[2], w[3]});
            p_new[1] = __builtin_bit_cast(bf16x8_t, u32x4_t{w[4], w[5], w[6], w[7]});
        };
        // a step whose results are moved back into the first of each pair
        auto step_a = [&](int it, int k0, const uint16_t* kp, const uint16_t* vp) __attribute__((always_inline)) {
            step(it, k0, kp, vp, s_a, s_b, p_a, p_b, std::integral_constant<int, 0>{});
            s_a = s_b;
            p_a[0] = p_b[0];
            p_a[1] = p_b[1];
        };
        // slot j of the walk: a step while the wave has items left, then once the P.V of its last item
        auto slot = [&](int j, int it, const uint16_t* kp, const uint16_t* vp) __attribute__((always_inline)) {
            if (j < n_it) step_a(it, 32 * j, kp, vp);
            else if (j == n_it && n_it > 0) drain(vp);
        };

        // tile t: the step of its first item, the barrier, K(t+2) and V(t+1) parked from sets KSET and VSET (which
        // are refilled with K(t+2+PF) and V(t+1+PF)), then the steps of its other items
        auto park_next = [&](int t, auto kset_c, auto vset_c, auto st_c) __attribute__((always_inline)) {
            constexpr int KSET = decltype(kset_c)::value;
            const int st = st_c;  // t & 1, as a constant where the caller knows it
            if constexpr (DIRECT) {
                // K(t+2) over K(t), V(t+1) over V(t-1): requested now that every wave is done with those, awaited
                // (vmcnt) ahead of the next tile's barrier
                // (BIAS: always, so that a step knows how many requests follow that for its bias values; behind the last
                // tiles they land zeros that nobody reads)
                if (BIAS || t + 2 < n_tiles) dl_tile(Kd, dl_k, dl_k_on, (uint32_t)(t + 2) * tile_bytes_g, (uint32_t)(st * STAGE_B));
                if (BIAS || t + 1 < n_tiles) dl_tile(Vd, dl_v, dl_v_on, (uint32_t)(t + 1) * tile_bytes_g, (uint32_t)((2 + (st ^ 1)) * STAGE_B));
            } else {
                // (behind the last tiles these park and request copies of the last tile, which nobody reads)
                park_k(kreg[KSET], st);
                park_v(vset_c, st ^ 1);
                issue_k(kreg[KSET], (t + 2 + PF) * KT);
                issue_v(vset_c, (t + 1 + PF) * KT);
            }
        };
        // what a wave does ahead of a tile's barrier: DIRECT waits for its own requests of a tile ago
        // (BIAS: all but those for bias values, the last the wave has made when `stepped` -- a step lies between them and
        // the tile's requests)
        auto meet = [&](auto stepped_c) __attribute__((always_inline)) {
            if constexpr (DIRECT && BIAS && decltype(stepped_c)::value) {
                asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  // (of a last item's sixteen pieces it waits for twelve)
            } else if constexpr (DIRECT) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            __syncthreads();
        };
        // the same for a tile of which the wave walks every item: straight-line code, the pairs swapped from step to step
        // `st_c` is t & 1, as an integer or as a compile-time constant: with the stage known at compile time every LDS
        // address of the tile is the lane's base plus an immediate, and `later` (t > 0 known) drops the choice of the
        // first tile's stand-in for V(-1)
        auto walk_full = [&](int t, auto kset_c, auto vset_c, auto st_c, auto later_c) __attribute__((always_inline)) {
            const int st = st_c;
            constexpr bool kLater = decltype(later_c)::value;
            const int k0 = t * KT;
            if (NI > 1) {
                step(0, k0, k_at(st, 1), (!kLater && t == 0) ? v_at(st, 0) : v_at(st ^ 1, NI - 1), s_a, s_b, p_a, p_b, std::integral_constant<int, 0>{});
                meet(std::true_type{});
                park_next(t, kset_c, vset_c, st_c);
                step(1, k0 + 32, k_at(st ^ 1, 0), v_at(st, 0), s_b, s_a, p_b, p_a, std::integral_constant<int, DIRECT ? 2 * NLD : 0>{});
            } else {
                step_a(0, k0, k_at(st ^ 1, 0), (!kLater && t == 0) ? v_at(st, 0) : v_at(st ^ 1, 0));
                __syncthreads();
                park_next(t, kset_c, vset_c, st_c);
                __syncthreads();
            }
            keep_cur = keep_next;
        };
        auto walk_tile = [&](int t, auto kset_c, auto vset_c) __attribute__((always_inline)) {
            const int st = t & 1;  // K(t) and V(t) sit in stage st, K(t+1) and V(t-1) in the other
            // first item: the next item is item 1 of this tile (or item 0 of the next tile when a tile is one item);
            // the previous item is the last of tile t - 1 (at t = 0 there is none: P is zero, and V(0) stands in)
            slot(t * NI, 0, NI > 1 ? k_at(st, 1) : k_at(st ^ 1, 0), t == 0 ? v_at(st, 0) : v_at(st ^ 1, NI - 1));
            meet(std::false_type{});
            park_next(t, kset_c, vset_c, st);
            if (NI > 1) {
                slot(t * NI + 1, 1, k_at(st ^ 1, 0), v_at(st, 0));
            } else {
                __syncthreads();  // one item per tile: K(t+2) is read by the very next step
            }
            keep_cur = keep_next;
        };
        int t0 = 0;  // t0 % PF == 0 throughout (DIRECT knows no sets): the set indices below are compile-time
        if constexpr (WIN && PIPE) {
            static_assert(!WIN || !PIPE || (DIRECT && NI == 2), "a window's pipelined walk moves its tiles straight to LDS");
            using IC0 = std::integral_constant<int, 0>;
            for (; t0 < j_first / NI; t0++) {
                meet(std::false_type{});
                park_next(t0, IC0{}, IC0{}, t0 & 1);
            }
            const int st = t0 & 1;
            if (j_first & 1) {
                first_scores(1, 32 * j_first, k_at(st, 1), s_b);
                meet(std::false_type{});
                park_next(t0, IC0{}, IC0{}, st);
                step(1, 32 * j_first, k_at(st ^ 1, 0), v_at(st, 0), s_b, s_a, p_b, p_a, IC0{});
                late_max(0, 32 * j_first + 32, s_a);
                t0++;
            } else if (n_it > 0) {
                first_scores(0, 32 * j_first, k_at(st, 0), s_a);
                if (n_it > j_first + 1) {  // (V of the tile itself has landed by the barrier only, but for tile 0)
                    step(0, 32 * j_first, k_at(st, 1), t0 == 0 ? v_at(0, 0) : v_at(st ^ 1, 1), s_a, s_b, p_a, p_b, IC0{});
                    meet(std::true_type{});
                    park_next(t0, IC0{}, IC0{}, st);
                    late_max(1, 32 * j_first + 32, s_b);
                    step(1, 32 * j_first + 32, k_at(st ^ 1, 0), v_at(st, 0), s_b, s_a, p_b, p_a, IC0{});
                    t0++;
                }
            }
        }
        if (!PIPE) {
            static_assert(PIPE || PF == 1, "the unpipelined walk keeps one register set");
            for (int t = 0; t < n_tiles; t++) {
                const int st = t & 1;
#pragma unroll
                for (int it = 0; it < NI; it++)
                    if (t * NI + it < n_it && t * NI + it >= j_first)
                        step_simple(it, t * KT + 32 * it, k_at(st, it), v_at(st, it));
                park_k(kreg[0], st ^ 1);
                park_v(std::integral_constant<int, 0>{}, st ^ 1);
                issue_k(kreg[0], (t + 2) * KT);
                issue_v(std::integral_constant<int, 0>{}, (t + 2) * KT);
                __syncthreads();
                keep_cur = keep_next;
            }
            t0 = n_tiles;
        }
        const int t_full = PIPE ? n_it / NI : 0;
        if constexpr (DIRECT && !BIAS) {
            // (the others have no register to spare for the second copy of the tile's code)  Tile 0 (under a window the one
            // behind the first where it is even) on its own, then the tiles in pairs (odd, even) whose LDS stages are
            // compile-time constants, then what is left of the tiles the wave walks in full
            using IC0 = std::integral_constant<int, 0>;
            using IC1 = std::integral_constant<int, 1>;
            if (PIPE && t0 < t_full && (!WIN || (t0 & 1) == 0)) {
                walk_full(WIN ? t0 : 0, IC0{}, IC0{}, IC0{}, std::integral_constant<bool, WIN>{});
                t0++;
            }
            for (; PIPE && t0 + 2 <= t_full; t0 += 2) {
                walk_full(t0, IC0{}, IC0{}, IC1{}, std::true_type{});
                walk_full(t0 + 1, IC0{}, IC0{}, IC0{}, std::true_type{});
            }
            if (PIPE && t0 < t_full) {
                walk_full(t0, IC0{}, IC0{}, t0 & 1, std::true_type{});
                t0++;
            }
        } else {
            for (; PIPE && t0 + PF <= t_full; t0 += PF) {
                walk_full(t0, std::integral_constant<int, 2 % PF>{}, std::integral_constant<int, 1 % PF>{}, t0 & 1, std::false_type{});
                if (PF >= 2) walk_full(t0 + 1, std::integral_constant<int, 3 % PF>{}, std::integral_constant<int, 2 % PF>{}, (t0 + 1) & 1, std::false_type{});
                if (PF >= 3) walk_full(t0 + 2, std::integral_constant<int, 4 % PF>{}, std::integral_constant<int, 3 % PF>{}, (t0 + 2) & 1, std::false_type{});
            }
        }
        for (; t0 < n_loop; t0 += PF) {
            walk_tile(t0, std::integral_constant<int, 2 % PF>{}, std::integral_constant<int, 1 % PF>{});
            if (PF >= 2 && t0 + 1 < n_loop) walk_tile(t0 + 1, std::integral_constant<int, 3 % PF>{}, std::integral_constant<int, 2 % PF>{});
            if (PF >= 3 && t0 + 2 < n_loop) walk_tile(t0 + 2, std::integral_constant<int, 4 % PF>{}, std::integral_constant<int, 3 % PF>{});
        }
        // a wave that walked every item of the workgroup still owes the last P.V
        if (PIPE && n_it == n_loop * NI && n_it > 0) drain(v_at((n_loop - 1) & 1, NI - 1));
        if constexpr (BIAS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (requests behind the last item and the last tile)
        __syncthreads();  // the output rows are staged over the tiles
        if constexpr (HALVES) {
            // the second half's O (relative to its running max), max and lane's share of the row sum, as the registers hold
            // them, over its tiles and behind the first half's output rows
            f32x4_t* const part_o = (f32x4_t*)(lds + kTilesLds + wave * (32 * DP * 4)) + lane;
            float* const part_ml = (float*)(lds + kTilesLds - 2048) + 128 * wave + lane;
            if (half) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        part_o[64 * (4 * dt + j)] = f32x4_t{acc_o[dt][4 * j], acc_o[dt][4 * j + 1], acc_o[dt][4 * j + 2], acc_o[dt][4 * j + 3]};
                part_ml[0] = m_run;
                part_ml[64] = l_run;
            }
            __syncthreads();
            if (half) return;
            const float m_1 = part_ml[0], l_1 = part_ml[64];
            const float m_new = t_vmax(m_run, m_1), m_use = m_new == neg_inf() ? 0.0f : m_new;
            const float a_0 = __builtin_amdgcn_exp2f((m_run - m_use) * cc), a_1 = __builtin_amdgcn_exp2f((m_1 - m_use) * cc);
            l_run = l_run * a_0 + l_1 * a_1;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const f32x4_t o_1 = part_o[64 * (4 * dt + j)];
#pragma unroll
                    for (int e = 0; e < 4; e++) acc_o[dt][4 * j + e] = acc_o[dt][4 * j + e] * a_0 + o_1[e] * a_1;
                }
        }
    } else if (HALVES && half) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }
    // (a workgroup without tiles still has its early requests in flight: they land in its LDS)
    if constexpr (DIRECT) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- output: acc_o[dt][4j + e] = O^T[d = 32dt + 8j + 4hh + e][row col of the wave].  A lane holds 8-byte pieces of
    // its row; the wave parks its 32 normalised rows in its own region of LDS (every wave is past the last
    // barrier, and the region's previous content was read by this wave alone) and streams them out as whole rows,
    // 16 bytes per lane.
    const float l = t_sum_with_other_half(l_run);
    if constexpr (SPLIT) {
        // The partial of this span: O as accumulated (relative to the running max as it stands), that max in the exp2
        // domain, the row sum.  A workgroup without tiles, or a row that saw no key of the span, leaves (0, -inf, 0).
        // Stored as it stands in the registers, 32 rows to a block: eight columns of the 32 rows are 1 KB in one piece
        // (row by row, 16 bytes here and there, the stores took 1-2 us of a short span).  Above head dim 64 they go out at device
        // scope, so that the end of the launch has no megabytes in the L2s to write back: us, 32 / 8 heads of 128, 64 positions
        // over 8192 keys 22.1 -> 21.3, 16 15.3 -> 15.05; 28 / 4 heads, 200 over 3000 26.6 -> 23.5.  (Past the caches: 23.3 there,
        // 17.1 for 16.5 with 3 positions of 5 sequences over 1109 keys of 256.)  At head dim 64 the partials are few enough for
        // the write-back to be the shorter way: 16 heads, 2 positions over 900 keys 10.1, 10.4 at device scope.
        constexpr int kPartScope = DP > 64 ? 16 : 0;  // sc1
        const int r = q0 + 32 * wq + col;
        if (r < rows_total) {
            const size_t block = (((size_t)b * p.kv_heads + kvh) * (size_t)((rows_total + 31) / 32) + (size_t)(q0 / 32 + wq)) * (size_t)p.n_splits + (size_t)split;
            const __amdgpu_buffer_rsrc_t po = __builtin_amdgcn_make_buffer_rsrc(p.part_o + block * (size_t)(32 * D), 0, 128u * (uint32_t)D, kBufferFlags);
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (32 * dt + 8 * j < D)
                        __builtin_amdgcn_raw_buffer_store_b128(
                            __builtin_bit_cast(u32x4_t, f32x4_t{acc_o[dt][4 * j], acc_o[dt][4 * j + 1], acc_o[dt][4 * j + 2], acc_o[dt][4 * j + 3]}), po,
                            16u * (uint32_t)lane, 1024u * (uint32_t)(4 * dt + j), kPartScope);
            p.part_ml[64 * block + lane] = hh == 0 ? m_run * cc : l;
        }
        return;
    }
    const bool good = (l > 0.0f) && (l < __uint_as_float(0x7f800000u)) && !poison;
    // the hardware reciprocal (1 ulp) instead of the division's dozen instructions: the output is rounded to bf16
    const float inv_l = __builtin_amdgcn_rcpf(l);
    // Packed rows are positions of a chunked decode: one that sees no key at all is a row of zeros, as the reference's
    // decode kernels leave it (crates/rustorch-metal/src/kernels.rs:14504-14514: every loop runs zero times), not the
    // NaN row of flash_forward's l > 0 test.  l == 0 exactly when no key was weighed (a visible key gives P >= 1).
    const float bad = (PACKED && l == 0.0f) ? 0.0f : quiet_nan();
    uint16_t* const obuf = (uint16_t*)(lds + wq * Cfg::REGION);
    const float fill = p.zero_padded_rows ? 0.0f : quiet_nan();
    if (n_loop > 0) {
        uint16_t* const orow = obuf + col * LDK + 4 * hh;
        if (__all(good && valid)) {
            // the common wave: one multiplication per element (a branch of its own: as a select inside one loop the
            // compiler kept three selects per element for every wave)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *(u32x2_t*)(orow + 32 * dt + 8 * j) =
                        u32x2_t{t_cvt_pk_bf16(acc_o[dt][4 * j] * inv_l, acc_o[dt][4 * j + 1] * inv_l),
                                t_cvt_pk_bf16(acc_o[dt][4 * j + 2] * inv_l, acc_o[dt][4 * j + 3] * inv_l)};
        } else {
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float x = good ? acc_o[dt][4 * j + e] * inv_l : bad;
                        if (!valid) x = fill;
                        o[e] = x;
                    }
                    *(u32x2_t*)(orow + 32 * dt + 8 * j) = u32x2_t{t_cvt_pk_bf16(o[0], o[1]), t_cvt_pk_bf16(o[2], o[3])};
                }
        }
    }
    // (the same wave wrote and now reads: no barrier needed, the LDS queue is in order)
    const uint32_t fill2 = t_cvt_pk_bf16(fill, fill);
    if constexpr (!PACKED && 64 % CH == 0 && (DP <= 128 || DIRECT)) {
        // rows of one head, and a wave's store instruction covers whole rows: lane l moves chunk l % CH of the rows
        // l / CH, l / CH + 64 / CH, ... -- one address, then a constant step
        constexpr int RS = 64 / CH;  // rows per store instruction
        const int row0 = (int)((unsigned)lane / (unsigned)CH), ch = (int)((unsigned)lane % (unsigned)CH);
        const int rr0 = q0 + 32 * wq + row0;
        uint16_t* dst = p.out + (size_t)b * p.lo.batch_stride + (size_t)h0 * p.lo.head_stride + (size_t)rr0 * p.lo.row_pitch + 8 * ch;
        const size_t step = (size_t)RS * (size_t)p.lo.row_pitch;
        const uint16_t* src = obuf + row0 * LDK + 8 * ch;
        const bool col_ok = 8 * ch < D;
#pragma unroll
        for (int n = 0; n < CH / 2; n++) {
            const int rr = rr0 + RS * n;
            // no key tile walked: padded rows get the fill value, valid rows (which then see no key at all) NaN
            const uint32_t f2 = rr < n_q ? 0x7fc07fc0u : fill2;
            u32x4_t val = {f2, f2, f2, f2};
            if (n_loop > 0) val = *(const u32x4_t*)(src + RS * n * LDK);
            if (rr < rows_total && col_ok) store_row(dst, val);
            dst += step;
        }
    } else {
#pragma unroll
        for (int n = 0; n < CH / 2; n++) {
            const int cidx = lane + 64 * n;
            const int row = cidx / CH, ch = cidx - row * CH;
            const int rr = q0 + 32 * wq + row;
            const int sp = G > 1 ? rr / G : rr;
            const int gg = rr - sp * G;
            // no key tile walked: padded rows get the fill value, valid rows (which then see no key at all) NaN -- zeros
            // when the rows are positions of a chunked decode
            const uint32_t f2 = sp < n_q ? (PACKED ? 0u : 0x7fc07fc0u) : fill2;
            u32x4_t val = {f2, f2, f2, f2};
            if (n_loop > 0) val = *(const u32x4_t*)(obuf + row * LDK + 8 * ch);
            if (rr < rows_total && 8 * ch < D) {
                uint16_t* dst = p.out + (size_t)b * p.lo.batch_stride + (size_t)(h0 + gg) * p.lo.head_stride +
                                (size_t)sp * p.lo.row_pitch + 8 * ch;
                store_row(dst, val);
            }
        }
    }
}

// Folds the partials the SPLIT kernel leaves: each is weighed by 2^(m - max m), o / l goes out as bf16 where the unsplit
// kernel would have written the row.  No partial with a key (every m is -inf): the position sees no key at all, a row
// of zeros.  A wave takes eight columns of 32 rows, as the partials hold them: 1 KB a load, and a lane's weights are its
// own row's.  With many partials the four waves of a workgroup share them out (PARTS) and meet in LDS: a wave has eight
// loads of each kind in flight, and a latency for every eight is what the kernel takes, beside what stands ahead of the
// first of them: the grid is (columns, row block, (sequence, kv head)) and the arguments are the kernel's own, so that
// no division and no second round of argument loads does; partials behind the last are zeros by the descriptor, no branch.  us
// of the whole call, before -> now, new positions over context: 32 / 8 heads of 128, 16 over 8192 14.76 -> 14.45, 4 x 8 over 1024 12.25 ->
// 11.62; 28 / 4 of 128, 4 over 300 8.75 -> 8.27; 2 x 16 / 2 of 256, 5 over 3000 15.73 -> 15.40.
struct SplitMergeParams {
    const float *part_o, *part_ml;
    int n, dim, blocks, rows;  // partials, head dim, blocks of 32 rows and rows of a (sequence, kv head)
    uint16_t* out;
    long long batch_stride, head_stride, row_pitch;
    int pack, kv_heads;
    uint32_t pack_magic, kv_magic;  // div_magic
};

template <bool PARTS>
__global__ __launch_bounds__(256) void flash_split_merge_kernel(SplitMergeParams p) {
    constexpr int kGroup = 8;
    __shared__ float fold[PARTS ? 3 : 1][6][64];
    const int D = p.dim, n = p.n, lane = threadIdx.x % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t piece = PARTS ? blockIdx.x : 4 * blockIdx.x + wave;
    asm volatile("" ::"s"(p.part_o), "s"(p.part_ml), "s"(n), "s"(D), "s"(p.blocks), "s"(p.out), "s"(p.batch_stride), "s"(p.head_stride), "s"(p.row_pitch), "s"(p.pack), "s"(p.kv_heads),
                 "s"(p.pack_magic), "s"(p.kv_magic), "s"(p.rows));  // (loaded in one go)
    if (!PARTS && piece >= (uint32_t)D / 8) return;
    const size_t block = (size_t)(blockIdx.z * (uint32_t)p.blocks + blockIdx.y) * (uint32_t)n;
    const uint32_t o_bytes = 128u * (uint32_t)D;
    const __amdgpu_buffer_rsrc_t ml = __builtin_amdgcn_make_buffer_rsrc((void*)(p.part_ml + block * 64), 0, (uint32_t)n * 256u, kBufferFlags);
    const __amdgpu_buffer_rsrc_t po = __builtin_amdgcn_make_buffer_rsrc((void*)(p.part_o + block * (uint32_t)(32 * D)), 0, (uint32_t)n * o_bytes, kBufferFlags);
    const uint32_t ml_lane = 4u * (uint32_t)(lane & 31), po_lane = 1024u * piece + 16u * (uint32_t)lane;

    constexpr int STEP = PARTS ? 4 : 1;
    float m_all = neg_inf(), l_all = 0.0f;
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    bool nan_m = false;
    int k0 = PARTS ? (int)wave : 0;  // (below n: PARTS comes with more than eight)
    do {
        float mv[kGroup], lv[kGroup];
        f32x4_t ov[kGroup];
#pragma unroll
        for (int j = 0; j < kGroup; j++) {
            const uint32_t k = (uint32_t)(k0 + STEP * j);
            mv[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ml, ml_lane + 256u * k, 0, 0));
            lv[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ml, ml_lane + 256u * k + 128u, 0, 0));
            ov[j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(po, po_lane + o_bytes * k, 0, 0));
        }
        __builtin_amdgcn_sched_barrier(0);  // (all on their way before the first is awaited)
#pragma unroll
        for (int j = 0; j < kGroup; j++)
            if (k0 + STEP * j >= n) mv[j] = neg_inf();
        float m_new = m_all;
#pragma unroll
        for (int j = 0; j < kGroup; j++) {
            m_new = fmaxf(m_new, mv[j]);
            nan_m |= mv[j] != mv[j];
        }
        const float m_use = m_new == neg_inf() ? 0.0f : m_new;
        const float rescale = m_all == neg_inf() ? 0.0f : __builtin_amdgcn_exp2f(m_all - m_use);
        l_all *= rescale;
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] *= rescale;
#pragma unroll
        for (int j = 0; j < kGroup; j++) {
            // an empty partial (m = -inf) is the identity
            const float w = mv[j] == neg_inf() ? 0.0f : __builtin_amdgcn_exp2f(mv[j] - m_use);
            l_all += lv[j] * w;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] += ov[j][e] * w;
        }
        m_all = m_new;
        k0 += kGroup * STEP;
    } while (k0 < n);
    if constexpr (PARTS) {
        if (wave > 0) {
            fold[wave - 1][0][lane] = nan_m ? __builtin_nanf("") : m_all;
            fold[wave - 1][1][lane] = l_all;
#pragma unroll
            for (int e = 0; e < 4; e++) fold[wave - 1][2 + e][lane] = acc[e];
        }
        __syncthreads();
        if (wave > 0) return;
        float m_new = m_all;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            m_new = fmaxf(m_new, fold[j][0][lane]);
            nan_m |= fold[j][0][lane] != fold[j][0][lane];
        }
        const float m_use = m_new == neg_inf() ? 0.0f : m_new;
        const float rescale = m_all == neg_inf() ? 0.0f : __builtin_amdgcn_exp2f(m_all - m_use);
        l_all *= rescale;
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] *= rescale;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const float mj = fold[j][0][lane], w = mj == neg_inf() ? 0.0f : __builtin_amdgcn_exp2f(mj - m_use);
            l_all += fold[j][1][lane] * w;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] += fold[j][2 + e][lane] * w;
        }
        m_all = m_new;
    }
    const int r = (int)blockIdx.y * 32 + (lane & 31), bk = (int)blockIdx.z;
    if (r >= p.rows) return;
    const int b = div_magic(bk, p.kv_magic), kvh = bk - b * p.kv_heads, s_pos = div_magic(r, p.pack_magic), g = r - s_pos * p.pack;
    uint16_t* const dst = p.out + (size_t)b * p.batch_stride + (size_t)(kvh * p.pack + g) * p.head_stride + (size_t)s_pos * p.row_pitch +
                          8 * piece + 4 * (lane >> 5);
    uint2 x = make_uint2(0u, 0u);
    if (m_all != neg_inf() || nan_m) {
        x.x = (uint32_t)f32_to_bf16_bits(acc[0] / l_all) | (uint32_t)f32_to_bf16_bits(acc[1] / l_all) << 16;
        x.y = (uint32_t)f32_to_bf16_bits(acc[2] / l_all) | (uint32_t)f32_to_bf16_bits(acc[3] / l_all) << 16;
    }
    *(uint2*)dst = x;
}

// ---------------------------------------------------------------------------------------------------------------
// The same walk with 64 query rows per wave (two blocks of 32), head dim 64, masks none / causal, rows of one head.
// At head dim 64 a 32-key item is only 8 matrix instructions per 32 rows: what paces the tile kernel there is the
// movement of a key tile (LDS parking, the workgroup barrier per tile) and the operand reads, which are the same
// whether a wave multiplies a fragment into one row block or two.  Here every K and V fragment read from LDS feeds
// two matrix instructions, a tile in LDS serves 256 query rows between two barriers, and a workgroup's set-up is
// spread over twice the rows.  Two workgroups share a CU (two O blocks, two score tiles and their operands).
constexpr int WROWS = 256;  // query rows per workgroup: four waves of 64

template <int MODE>
__global__ __launch_bounds__(256, 2) void flash_wide_bf16_kernel(FlashTileParams p) {
    constexpr int DP = 64, KT = 64, LDK = DP + 8, LDV = DP + 32, NI = KT / 32, KS = DP / 16, DT = DP / 32, CH = DP / 8;
    constexpr int TTHREADS = 256, NL = KT * CH / TTHREADS, RB = 2;
    constexpr bool kCausal = MODE == kMaskCausal;
    constexpr int TILE_BYTES = 2 * KT * (LDK + LDV) * 2;  // two stages of K and V
    constexpr int REGION = 64 * LDK * 2;                  // a wave's staged output rows
    static_assert(4 * REGION <= TILE_BYTES, "the staged output rows fit over the tiles");
    static_assert(NI == 2 && KS == 2 * DT, "two items per tile, one P.V instruction per score instruction");

    __shared__ __attribute__((aligned(16))) unsigned char lds[TILE_BYTES];
    uint16_t* const Ks = (uint16_t*)lds;                 // [2][KT * LDK]
    uint16_t* const Vs = (uint16_t*)lds + 2 * KT * LDK;  // [2][KT * LDV]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    const int rows_total = p.seq_q;
    const int b = blockIdx.y;
    const int gx = (int)__umulhi(blockIdx.x, p.kv_magic);  // (as in the tile kernel)
    const int kvh = (int)blockIdx.x - gx * p.kv_heads, hx = kvh * p.group + gx;
    const uint16_t* const Kg = p.k + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;
    const uint16_t* const Vg = p.v + (size_t)b * p.lkv.batch_stride + (size_t)kvh * p.lkv.head_stride;

    // ---- tile movement, as in the tile kernel: chunk c = tid + 256 n of a tile is (row c / CH, 16-byte chunk c % CH)
    u32x4_t kreg[NL], vreg[NL], k1[NL];
    uint32_t ld_off[NL], st_k[NL], st_v[NL];
    const uint32_t kv_pitch = (uint32_t)p.lkv.row_pitch;
#pragma unroll
    for (int n = 0; n < NL; n++) {
        const int c = tid + TTHREADS * n;
        const int row = c / CH, ch = c - row * CH;
        st_k[n] = (uint32_t)((row * LDK + 8 * ch) * 2);
        st_v[n] = (uint32_t)((2 * KT * LDK + row * LDV + 8 * ch) * 2);
        ld_off[n] = ((uint32_t)row * kv_pitch + (uint32_t)(8 * ch)) * 2u;
    }
    const uint32_t tile_bytes_g = (uint32_t)KT * kv_pitch * 2u;
    {  // tile 0 (K and V) and K of tile 1, before the lengths have arrived: descriptors that end with the tensor
        const uint32_t all_bytes = p.seq_kv > 0 ? ((uint32_t)(p.seq_kv - 1) * kv_pitch + (uint32_t)DP) * 2u : 0u;
        const __amdgpu_buffer_rsrc_t Kall = __builtin_amdgcn_make_buffer_rsrc((void*)Kg, 0, all_bytes, kBufferFlags);
        const __amdgpu_buffer_rsrc_t Vall = __builtin_amdgcn_make_buffer_rsrc((void*)Vg, 0, all_bytes, kBufferFlags);
#pragma unroll
        for (int n = 0; n < NL; n++) {
            kreg[n] = __builtin_amdgcn_raw_buffer_load_b128(Kall, ld_off[n], 0, 0);
            vreg[n] = __builtin_amdgcn_raw_buffer_load_b128(Vall, ld_off[n], 0, 0);
            k1[n] = __builtin_amdgcn_raw_buffer_load_b128(Kall, ld_off[n], tile_bytes_g, 0);
        }
    }

    const int n_q = p.q_lens ? min(max(p.q_lens[b], 0), p.seq_q) : p.seq_q;          // valid query positions
    const int n_keys = p.kv_lens ? min(max(p.kv_lens[b], 0), p.seq_kv) : p.seq_kv;  // keys that exist
    // rank of the query tile: the last one first; in a padded batch counted from the sequence's own last valid tile
    int qtile = p.n_qtiles - 1 - (int)blockIdx.z;
    if (p.q_lens) {
        const int n_qt = (n_q + WROWS - 1) / WROWS;
        const int rank = (int)blockIdx.z;
        qtile = rank < n_qt ? n_qt - 1 - rank : rank;
    }
    const int q0 = qtile * WROWS;
    const int wq = (wave + hx + b + (int)blockIdx.z) & 3;  // which 64 rows of the tile: rotated, as in the tile kernel
    const int r0 = q0 + 64 * wq;                           // the wave's first row
    const int off = n_keys - n_q;                          // causal: the last valid query sees every key

    int kv_end = n_keys;
    if (kCausal) kv_end = min(n_keys, min(q0 + WROWS - 1, n_q - 1) + off + 1);
    if (q0 >= n_q) kv_end = 0;
    kv_end = max(kv_end, 0);
    const int n_tiles = (kv_end + KT - 1) / KT;

    const uint32_t fill2 = p.zero_padded_rows ? 0u : 0x7fc07fc0u;
    if (q0 >= n_q) {  // padded rows only: the fill value, and done
        const u32x4_t val = {fill2, fill2, fill2, fill2};
        uint16_t* const ob = p.out + (size_t)b * p.lo.batch_stride + (size_t)hx * p.lo.head_stride;
        for (int c = tid; c < WROWS * CH; c += TTHREADS) {
            const int row = c / CH, ch = c - row * CH;
            if (q0 + row < rows_total) *(u32x4_t*)(ob + (size_t)(q0 + row) * p.lo.row_pitch + 8 * ch) = val;
        }
        return;
    }
    // descriptors that end with the last key's row: rows behind it come back as zeros
    const uint32_t slab_bytes = n_keys > 0 ? ((uint32_t)(n_keys - 1) * kv_pitch + (uint32_t)DP) * 2u : 0u;
    const __amdgpu_buffer_rsrc_t Kbuf = __builtin_amdgcn_make_buffer_rsrc((void*)Kg, 0, slab_bytes, kBufferFlags);
    const __amdgpu_buffer_rsrc_t Vbuf = __builtin_amdgcn_make_buffer_rsrc((void*)Vg, 0, slab_bytes, kBufferFlags);
    if (n_keys < KT) {  // the early requests ended with the tensor, not with the sequence
#pragma unroll
        for (int n = 0; n < NL; n++)
            if ((tid + TTHREADS * n) / CH >= n_keys) vreg[n] = u32x4_t{0u, 0u, 0u, 0u};
    }

    f32x16_t acc_o[RB][DT];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc_o[rb][t][i] = 0.0f;
    float m_run[RB], l_run[RB];
    bool valid[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        m_run[rb] = neg_inf();
        l_run[rb] = 0.0f;
        valid[rb] = false;
    }
    const float cc = p.scale_log2e;  // exp2 argument per unit of score

    if (n_tiles > 0) {
        const int last_kv0 = (n_tiles - 1) * KT;
        auto issue_k = [&](int kv0) __attribute__((always_inline)) {
            const uint32_t tile_off = (uint32_t)min(kv0, last_kv0) * (kv_pitch * 2u);
#pragma unroll
            for (int n = 0; n < NL; n++) kreg[n] = __builtin_amdgcn_raw_buffer_load_b128(Kbuf, ld_off[n], tile_off, 0);
        };
        auto issue_v = [&](int kv0) __attribute__((always_inline)) {
            const uint32_t tile_off = (uint32_t)min(kv0, last_kv0) * (kv_pitch * 2u);
#pragma unroll
            for (int n = 0; n < NL; n++) vreg[n] = __builtin_amdgcn_raw_buffer_load_b128(Vbuf, ld_off[n], tile_off, 0);
        };
        auto park_k = [&](const u32x4_t (&src)[NL], int st) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NL; n++) *(u32x4_t*)(lds + st * (KT * LDK * 2) + st_k[n]) = src[n];
        };
        auto park_v = [&](int st) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NL; n++) *(u32x4_t*)(lds + st * (KT * LDV * 2) + st_v[n]) = vreg[n];
        };

        // ---- this lane's two query rows, and the wave's limits as scalars
        int lim[RB], wave_lim_min[RB];
        const int r_lim = min(rows_total, n_q);  // rows below it are valid
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const int r = r0 + 32 * rb + col;
            valid[rb] = r < r_lim;
            int l = n_keys - 1;  // last key this row sees
            if (kCausal) l = min(l, r + off);
            lim[rb] = valid[rb] ? l : -1;
            const int r_first = r0 + 32 * rb, r_last = r_first + 31;
            wave_lim_min[rb] = r_last < r_lim ? (kCausal ? min(n_keys - 1, r_first + off) : n_keys - 1) : -1;
        }
        const int r_top = min(r0 + 63, r_lim - 1);
        const int wave_lim_max = r0 < r_lim ? (kCausal ? min(n_keys - 1, r_top + off) : n_keys - 1) : -1;
        // items this wave walks: the ones that hold a key some row of it sees (a prefix of the workgroup's items)
        const int n_it = wave_lim_max < 0 ? 0 : min(n_tiles * NI, (wave_lim_max >> 5) + 1);

        // ---- Q as B operands: column q = lane % 32 of either row block, contraction slots 16 ks + 8 hh .. + 8
        bf16x8_t qreg[RB][KS];
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const int r_q = min(r0 + 32 * rb + col, rows_total - 1);  // (a row past the tensor reads the last row: it is masked and not written)
            const size_t q_off = (size_t)b * p.lq.batch_stride + (size_t)hx * p.lq.head_stride + (size_t)r_q * p.lq.row_pitch;
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                qreg[rb][ks] = __builtin_bit_cast(bf16x8_t, *(const u32x4_t*)(p.q + q_off + 16 * ks + 8 * hh));
        }
        const int k_off = col * LDK + 8 * hh;
        const int v_off = (((lane & 15) >> 2) + 4 * hh) * LDV + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

        // K(0), V(0) -> stage 0, K(1) -> stage 1; the register sets then take K(2) and V(1)
        park_k(kreg, 0);
        park_v(0);
        park_k(k1, 1);
        issue_k(2 * KT);
        issue_v(KT);
        __syncthreads();

        auto mask_item = [&](int rb, int k0, f32x16_t& sc) __attribute__((always_inline)) {
            if (k0 + 31 > wave_lim_min[rb]) {
                const int room = lim[rb] - k0 - 4 * hh;  // key k0 + 8 (i / 4) + 4 hh + i % 4 is hidden when it lies past lim
#pragma unroll
                for (int i = 0; i < 16; i++) sc[i] = (8 * (i >> 2) + (i & 3) > room) ? neg_inf() : sc[i];
            }
        };
        auto load_v = [&](int i, const uint16_t* vp) __attribute__((always_inline)) {
            const int u = i / DT, dt = i - u * DT;
            const u32x2_t lo = t_lds_read_tr16(vp + 16 * u * LDV + 32 * dt);
            const u32x2_t hi = t_lds_read_tr16(vp + 16 * u * LDV + 32 * dt + 8 * LDV);
            return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        };
        auto pin_f = [](float& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
        auto pin_u = [](uint32_t& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
        auto pin_b = [](bf16x8_t& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };

        float neg_mc[RB];  // -m_run * cc; +inf while a valid row has no max yet
        f32x16_t s_a[RB];                 // S(j), made at the end of step j - 1
        bf16x8_t p_a[RB][2], p_b[RB][2];  // P(j - 1) and P(j)
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            neg_mc[rb] = valid[rb] ? __uint_as_float(0x7f800000u) : 0.0f;
            p_a[rb][0] = p_a[rb][1] = p_b[rb][0] = p_b[rb][1] = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
#pragma unroll
            for (int i = 0; i < 16; i++) s_a[rb][i] = 0.0f;
        }
        // S(0), and the running max started from it, so that the first step already runs the fast path
        if (n_it > 0) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const bf16x8_t kf = *(const bf16x8_t*)(Ks + k_off + 16 * ks);
#pragma unroll
                for (int rb = 0; rb < RB; rb++) s_a[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qreg[rb][ks], s_a[rb], 0, 0, 0);
            }
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                mask_item(rb, 0, s_a[rb]);  // (the step applies the mask again, which changes nothing)
                const float m0 = t_max_with_other_half(t_max16(s_a[rb]));
                if (m0 > neg_inf()) {  // (false for -inf and for NaN: such a row waits for the slow path)
                    m_run[rb] = m0;
                    neg_mc[rb] = -m0 * cc;
                }
            }
        }

        // O^T += V(j-1)^T . P(j-1)^T alone: behind the wave's last item
        auto drain = [&](const uint16_t* vp) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const int u = i / DT, dt = i - u * DT;
                const bf16x8_t av = __builtin_bit_cast(bf16x8_t, load_v(i, vp));
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
                    acc_o[rb][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, p_a[rb][u], acc_o[rb][dt], 0, 0, 0);
            }
        };
        auto exp_plain = [&](const f32x16_t& sc, float nmc, uint32_t (&w)[8], float& part) __attribute__((always_inline)) {
            float part0 = 0.0f, part1 = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * e], cc, nmc));
                const float x1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * e + 1], cc, nmc));
                part0 += x0;
                part1 += x1;
                w[e] = t_cvt_pk_bf16(x0, x1);
            }
            part = part0 + part1;
        };
        // the slow path of a softmax step: the item max, O and l rescaled to it, P again from the scores
        auto raise_max_and_redo = [&](int rb, const f32x16_t& sc, uint32_t (&w)[8], float& part) __attribute__((always_inline)) {
            const float m_item = t_max_with_other_half(t_max16(sc));
            const float m_new = t_vmax(m_run[rb], m_item);
            const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
            const float alpha = __builtin_amdgcn_exp2f((m_run[rb] - m_use) * cc);  // m_run = -inf -> 0
            m_run[rb] = m_new;
            l_run[rb] *= alpha;
#pragma unroll
            for (int tt = 0; tt < DT; tt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc_o[rb][tt][i] *= alpha;
            const float mc = m_use * cc;
            neg_mc[rb] = (m_new == neg_inf()) ? (valid[rb] ? __uint_as_float(0x7f800000u) : 0.0f) : -mc;
            exp_plain(sc, -mc, w, part);
        };

        // One step: item j (keys k0 ..) gets its softmax step in both row blocks; K rows of item j + 1 are at kp, V rows
        // of item j - 1 at vp.  The registers hold one score tile per row block (two workgroups per CU), so the row
        // blocks are staggered: while block 0's P(j) is made its P.V instructions of item j - 1 run; while block 1's
        // P(j) is made, block 1's P.V instructions and block 0's S(j+1) run (into the registers block 0's S(j) has
        // just left); block 1's S(j+1) follows, and is still in flight when the next step starts on block 0.  Every V
        // and K fragment is read from LDS once and feeds both row blocks.  No row max in the steady state (see the
        // tile kernel).
        auto step = [&](int k0, const uint16_t* kp, const uint16_t* vp, bf16x8_t (&p_prev)[RB][2],
                        bf16x8_t (&p_new)[RB][2]) __attribute__((always_inline)) {
            mask_item(0, k0, s_a[0]);
            u32x4_t vop[KS], kop[KS];
            constexpr int PER = 16 / KS;  // scores of a row block per group
            const f32x16_t zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            // the vector work of group g of row block rb: a quarter of P(j), fenced
            auto quarter = [&](int rb, int g, float (&part)[2], uint32_t (&w)[8]) __attribute__((always_inline)) {
                float t[PER];
#pragma unroll
                for (int i = 0; i < PER; i++) t[i] = __builtin_fmaf(s_a[rb][PER * g + i], cc, neg_mc[rb]);
#pragma unroll
                for (int i = 0; i < PER; i++) t[i] = __builtin_amdgcn_exp2f(t[i]);
#pragma unroll
                for (int i = 0; i < PER; i += 2) {
                    part[0] += t[i];
                    part[1] += t[i + 1];
                    w[(PER * g + i) / 2] = t_cvt_pk_bf16(t[i], t[i + 1]);
                }
#pragma unroll
                for (int i = 0; i < PER; i++) pin_f(t[i]);
                pin_f(part[0]);
                pin_f(part[1]);
#pragma unroll
                for (int i = 0; i < PER; i += 2) pin_u(w[(PER * g + i) / 2]);
            };
            auto finish = [&](int rb, float (&part)[2], uint32_t (&w)[8]) __attribute__((always_inline)) {
                float pt = part[0] + part[1];
                if (__builtin_expect(__any(!(pt <= kTileTrigSum)), 0)) raise_max_and_redo(rb, s_a[rb], w, pt);
                l_run[rb] += pt;
                p_new[rb][0] = __builtin_bit_cast(bf16x8_t, u32x4_t{w[0], w[1], w[2], w[3]});
                p_new[rb][1] = __builtin_bit_cast(bf16x8_t, u32x4_t{w[4], w[5], w[6], w[7]});
            };
            // ---- row block 0: P(j), with its P.V of item j - 1
            {
                float part[2] = {0.0f, 0.0f};
                uint32_t w[8];
                vop[0] = load_v(0, vp);
#pragma unroll
                for (int g = 0; g < KS; g++) {
                    if (g + 1 < KS) vop[g + 1] = load_v(g + 1, vp);
                    const int u = g / DT, dt = g - u * DT;
                    acc_o[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vop[g]), p_prev[0][u], acc_o[0][dt], 0, 0, 0);
                    quarter(0, g, part, w);
                    pin_b(p_prev[0][u]);
                }
                finish(0, part, w);
            }
            // ---- row block 1: P(j), with its P.V of item j - 1 and row block 0's S(j+1)
            {
                mask_item(1, k0, s_a[1]);
                float part[2] = {0.0f, 0.0f};
                uint32_t w[8];
                kop[0] = *(const u32x4_t*)(kp);
#pragma unroll
                for (int g = 0; g < KS; g++) {
                    if (g + 1 < KS) kop[g + 1] = *(const u32x4_t*)(kp + 16 * (g + 1));
                    const int u = g / DT, dt = g - u * DT;
                    acc_o[1][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vop[g]), p_prev[1][u], acc_o[1][dt], 0, 0, 0);
                    s_a[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kop[g]), qreg[0][g], g == 0 ? zero16 : s_a[0], 0, 0, 0);
                    quarter(1, g, part, w);
                    pin_b(p_prev[1][u]);
                    pin_b(qreg[0][g]);
                }
                finish(1, part, w);
            }
            // ---- row block 1's S(j+1)
#pragma unroll
            for (int g = 0; g < KS; g++)
                s_a[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kop[g]), qreg[1][g], g == 0 ? zero16 : s_a[1], 0, 0, 0);
        };
        // a step whose results are moved back into the first of each pair
        auto step_a = [&](int k0, const uint16_t* kp, const uint16_t* vp) __attribute__((always_inline)) {
            step(k0, kp, vp, p_a, p_b);
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                p_a[rb][0] = p_b[rb][0];
                p_a[rb][1] = p_b[rb][1];
            }
        };
        // slot j of the walk: a step while the wave has items left, then once the P.V of its last item
        auto slot = [&](int j, const uint16_t* kp, const uint16_t* vp) __attribute__((always_inline)) {
            if (j < n_it) step_a(32 * j, kp, vp);
            else if (j == n_it && n_it > 0) drain(vp);
        };
        // behind the barrier of tile t: K(t+2) and V(t+1) parked over K(t) and V(t-1), K(t+3) and V(t+2) requested
        auto park_next = [&](int t, int st) __attribute__((always_inline)) {
            park_k(kreg, st);
            park_v(st ^ 1);
            issue_k((t + 3) * KT);
            issue_v((t + 2) * KT);
        };
        // a tile of which the wave walks both items: straight-line code, the pairs swapped from step to step
        auto walk_full = [&](int t, auto st_c, auto later_c) __attribute__((always_inline)) {
            const int st = st_c;
            constexpr bool kLater = decltype(later_c)::value;
            const uint16_t* const k_st = Ks + st * KT * LDK + k_off;
            const uint16_t* const k_ot = Ks + (st ^ 1) * KT * LDK + k_off;
            const uint16_t* const v_st = Vs + st * KT * LDV + v_off;
            const uint16_t* const v_ot = Vs + (st ^ 1) * KT * LDV + v_off;
            const int k0 = t * KT;
            step(k0, k_st + 32 * LDK, (!kLater && t == 0) ? v_st : v_ot + 32 * LDV, p_a, p_b);
            __syncthreads();
            park_next(t, st);
            step(k0 + 32, k_ot, v_st, p_b, p_a);
        };
        auto walk_tile = [&](int t) __attribute__((always_inline)) {
            const int st = t & 1;
            const uint16_t* const k_st = Ks + st * KT * LDK + k_off;
            const uint16_t* const k_ot = Ks + (st ^ 1) * KT * LDK + k_off;
            const uint16_t* const v_st = Vs + st * KT * LDV + v_off;
            const uint16_t* const v_ot = Vs + (st ^ 1) * KT * LDV + v_off;
            slot(t * NI, k_st + 32 * LDK, t == 0 ? v_st : v_ot + 32 * LDV);
            __syncthreads();
            park_next(t, st);
            slot(t * NI + 1, k_ot, v_st);
        };
        using IC0 = std::integral_constant<int, 0>;
        using IC1 = std::integral_constant<int, 1>;
        const int t_full = n_it / NI;
        int t0 = 0;
        if (t0 < t_full) {
            walk_full(0, IC0{}, std::false_type{});
            t0 = 1;
        }
        for (; t0 + 2 <= t_full; t0 += 2) {
            walk_full(t0, IC1{}, std::true_type{});
            walk_full(t0 + 1, IC0{}, std::true_type{});
        }
        if (t0 < t_full) {
            walk_full(t0, t0 & 1, std::true_type{});
            t0++;
        }
        for (; t0 < n_tiles; t0++) walk_tile(t0);
        // a wave that walked every item of the workgroup still owes the last P.V
        if (n_it == n_tiles * NI && n_it > 0) drain(Vs + ((n_tiles - 1) & 1) * KT * LDV + v_off + 32 * LDV);
        __syncthreads();  // the output rows are staged over the tiles
    }

    // ---- output: the wave parks its 64 normalised rows in its own region of LDS and streams them out as whole rows
    uint16_t* const obuf = (uint16_t*)(lds + wq * REGION);
    const float fill = p.zero_padded_rows ? 0.0f : quiet_nan();
    if (n_tiles > 0) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const float l = t_sum_with_other_half(l_run[rb]);
            const bool good = (l > 0.0f) && (l < __uint_as_float(0x7f800000u));
            const float inv_l = __builtin_amdgcn_rcpf(l);
            uint16_t* const orow = obuf + (32 * rb + col) * LDK + 4 * hh;
            if (__all(good && valid[rb])) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        *(u32x2_t*)(orow + 32 * dt + 8 * j) =
                            u32x2_t{t_cvt_pk_bf16(acc_o[rb][dt][4 * j] * inv_l, acc_o[rb][dt][4 * j + 1] * inv_l),
                                    t_cvt_pk_bf16(acc_o[rb][dt][4 * j + 2] * inv_l, acc_o[rb][dt][4 * j + 3] * inv_l)};
            } else {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        float o[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            float x = good ? acc_o[rb][dt][4 * j + e] * inv_l : quiet_nan();
                            if (!valid[rb]) x = fill;
                            o[e] = x;
                        }
                        *(u32x2_t*)(orow + 32 * dt + 8 * j) = u32x2_t{t_cvt_pk_bf16(o[0], o[1]), t_cvt_pk_bf16(o[2], o[3])};
                    }
            }
        }
    }
    // (the same wave wrote and now reads: no barrier needed, the LDS queue is in order)
    {
        constexpr int RS = 64 / CH;  // rows per store instruction
        const int row0 = lane / CH, ch = lane % CH;
        const int rr0 = r0 + row0;
        uint16_t* dst = p.out + (size_t)b * p.lo.batch_stride + (size_t)hx * p.lo.head_stride + (size_t)rr0 * p.lo.row_pitch + 8 * ch;
        const size_t step_e = (size_t)RS * (size_t)p.lo.row_pitch;
        const uint16_t* src = obuf + row0 * LDK + 8 * ch;
#pragma unroll
        for (int n = 0; n < 64 / RS; n++) {
            const int rr = rr0 + RS * n;
            // no key tile walked: padded rows get the fill value, valid rows (which then see no key at all) NaN
            const uint32_t f2 = rr < n_q ? 0x7fc07fc0u : fill2;
            u32x4_t val = {f2, f2, f2, f2};
            if (n_tiles > 0) val = *(const u32x4_t*)(src + RS * n * LDK);
            if (rr < rows_total) *(u32x4_t*)dst = val;
            dst += step_e;
        }
    }
}

// Output rows past the caches (store_past), up to head dim 128?  The call is never longer for it, but what it gains by not waiting
// for the write-back the kernel that reads the rows next pays in part, or, where they would have stayed in the L2s for it, in
// full and more.  us, plainly / past, the call, and it with a product of its rows and a [heads * dim, heads * dim] matrix behind it, by
// MB written: 1 (1 16 512 64) 8.57 / 8.56, 25.2 / 25.2; 2 (1 32/8 256 128) 8.38 / 8.38, 30.5 / 31.4; 4 (masked 2 16 1024 64) 17.7 / 17.5, 29.6 /
// 30.9, (window 300, 2 16 2000 32) 13.2 / 12.8, 24.0 / 25.3; 5 (window 256, 1 16 2500 64) 12.0 / 11.6, 24.6 / 25.9; 5.7 (2 16 700 80) 16.0 / 15.9,
// 29.0 / 30.7; 6.5 (1 40/8 640 128) 14.9 / 14.4, 61.1 / 61.0; 8 (1 32/8 1024 128) 19.7 / 18.8, 59.1 / 58.7, (window 256, 2 16 2048 64) 13.2 / 12.6,
// 27.7 / 27.9; 24 (2 32/8 1501 128) 45.3 / 44.5, 132.7 / 133.3; 32 (window 256, 4 16 4096 64) 41.0 / 39.2, 79.8 / 79.8, (padded, 16 16 1024 64)
// 28.2 / 26.2, 82.4 / 81.9; 48 (2 32/8 3000 128) 148.9 / 145.5, 315.6 / 319.1.  From 6 MB on the call gains 1 to 8 % and the two together are level;
// below, the two together lose up to 6 % for a call that gains up to 4.  Two kernels (PAST): where one chose by a branch around its
// stores, 2 32/8 1501 128 took 45.9 for 45.6, small calls with a branch a store 2 to 4 % longer.  Above head dim 128 without the choice: plainly
// under a window (4 40/8 2653 256 window 476 425 us, past the caches 437), past the caches otherwise (1 8/2 1024 256 46.9 -> 46.7).
static bool out_goes_past(const FlashTileParams& p) {
    const double written = 2.0 * p.batch * p.heads * (double)p.seq_q * p.dim;
    return written > 6.0 * (1 << 20);
}

template <int DP, int MODE, bool BIAS, bool PACKED, bool SPLIT = false, bool WIN = false, int TILES = kTilesRegs, bool HALVES = false, bool QROWS = true>
hipError_t launch_one(hipStream_t stream, const FlashTileParams& p, dim3 grid) {
    const dim3 block(HALVES ? 512 : TileCfg<DP>::THREADS);
    if constexpr (DP > 128) {
        hipLaunchKernelGGL((flash_tile_bf16_kernel<DP, MODE, BIAS, PACKED, SPLIT, WIN, TILES, HALVES, QROWS, !SPLIT && !WIN>), grid, block, 0, stream, p);
    } else if (!SPLIT && out_goes_past(p)) {  // (a span leaves partials)
        hipLaunchKernelGGL((flash_tile_bf16_kernel<DP, MODE, BIAS, PACKED, SPLIT, WIN, TILES, HALVES, QROWS, !SPLIT>), grid, block, 0, stream, p);
    } else {
        hipLaunchKernelGGL((flash_tile_bf16_kernel<DP, MODE, BIAS, PACKED, SPLIT, WIN, TILES, HALVES, QROWS, false>), grid, block, 0, stream, p);
    }
    return hipGetLastError();
}

template <int DP, int TILES>
hipError_t launch_packed(hipStream_t stream, const FlashTileParams& p, dim3 grid) {
    if (p.n_splits > 1) {  // (rows packed over a group of one head are rows of that head)
        hipError_t e = launch_one<DP, kMaskCausal, false, true, true, false, TILES>(stream, p, grid);
        if (e != hipSuccess) return e;
        auto magic = [](int d) { return d > 1 ? (uint32_t)(0x100000000ull / (unsigned)d) + 1u : 0u; };
        const int rows = p.seq_q * p.pack, blocks = (rows + 31) / 32, pieces = p.dim / 8;
        const SplitMergeParams m{p.part_o, p.part_ml, p.n_splits, p.dim, blocks, rows, p.out, p.lo.batch_stride, p.lo.head_stride, p.lo.row_pitch,
                                 p.pack, p.kv_heads, magic(p.pack), magic(p.kv_heads)};
        const dim3 at((unsigned)(p.n_splits > 8 ? pieces : (pieces + 3) / 4), (unsigned)blocks, (unsigned)(p.batch * p.kv_heads));
        if (p.n_splits > 8) hipLaunchKernelGGL(flash_split_merge_kernel<true>, at, dim3(256), 0, stream, m);
        else hipLaunchKernelGGL(flash_split_merge_kernel<false>, at, dim3(256), 0, stream, m);
        return hipGetLastError();
    }
    return launch_one<DP, kMaskCausal, false, true, false, false, TILES>(stream, p, grid);
}
template <int DP, int TILES>
hipError_t launch_tiles(hipStream_t stream, const FlashTileParams& p, dim3 grid) {
    if (p.n_splits > 1 || p.pack > 1 || p.decode_rows) return launch_packed<DP, TILES>(stream, p, grid);
    if (p.window > 0) return launch_one<DP, kMaskCausal, false, false, false, true, TILES>(stream, p, grid);
    if constexpr (DP > 128 && TILES != kTilesRegs) {
        if (p.bias) return hipErrorInvalidValue;  // (takes_tiles_direct)
    } else if (p.bias) {
        if (DP == 64 && (unsigned long long)grid.x * grid.y * grid.z > 2ull * (unsigned long long)p.n_cus)
            return launch_one<DP, kMaskNone, true, false, false, false, TILES, false, DP != 64>(stream, p, grid);
        return launch_one<DP, kMaskNone, true, false, false, false, TILES>(stream, p, grid);
    }
    if (p.mask == kMaskNone) return launch_one<DP, kMaskNone, false, false, false, false, TILES>(stream, p, grid);
    if (p.mask == kMaskCausal) return launch_one<DP, kMaskCausal, false, false, false, false, TILES>(stream, p, grid);
    return hipErrorInvalidValue;
}
// Two halves of the walk (head dims 64 and 128 exactly, up to 32, and 65 to 96): where every workgroup has a CU to itself and
// the walk is long enough to pay for the meeting at its end, 0.6-1.4 us.  us, whole / halves, B H N head dim: causal 1 8 384
// 64 8.0 / 8.1, 512 9.3 / 9.1, 1024 14.7 / 13.0, 4096 46.2 / 37.4; 1 8 256 128 8.8 / 10.3, 512 12.5 / 13.0, 1024 20.1 / 19.0,
// 4096 63.9 / 54.3; 1 8 512 96 10.4 / 10.7; unmasked 1 12 1000 96 19.5 / 17.4; 1 8 3000 32 37.2 / 28.2; with a bias 1 8 256 64
// 7.8 / 7.8, 512 11.5 / 10.3; 77 queries over 3001 keys, 24 heads of 32, 65.8 / 43.1.
constexpr int kHalvesFrom64 = 512, kHalvesFrom = 768;  // keys, head dims up to 64 and above
template <int DP, int TILES>
hipError_t launch_halves(hipStream_t stream, const FlashTileParams& p, dim3 grid) {
    if (p.bias) return launch_one<DP, kMaskNone, true, false, false, false, TILES, true>(stream, p, grid);
    if (p.mask == kMaskNone) return launch_one<DP, kMaskNone, false, false, false, false, TILES, true>(stream, p, grid);
    return launch_one<DP, kMaskCausal, false, false, false, false, TILES, true>(stream, p, grid);
}
// Up to 1.9 causal workgroups a CU: the long tiles are dispatched first, so that a long walk in halves and a short one behind
// it take a CU no longer than the longest walk whole, with its neighbour beside it -- from as many query tiles on as pay for
// two meetings a CU, and above head dim 64 from more where the heads do not divide by the eight XCDs and one gets more of the
// long tiles, where the heads of one tile number take more than an eighth of the CUs and the second round starts among tiles
// half as long as the longest, or where nearly every CU takes two.  us, whole / halves, causal, inputs that change from pass
// to pass, B H N: head dim 128 1 24 1300 29.2 / 27.0, 1 32 1523 36.8 / 33.3, 1 32 1684 40.2 / 39.5, 1 24 2150 48.6 / 42.2,
// 1 26 2246 53.4 / 51.9, 2 8 3612 76.8 / 65.7, but 5 8 1300 32.5 / 35.2, 5 8 1400 35.7 / 36.2, 4 12 1276 33.9 / 37.8, 1 28 2048
// 42.2 / 43.7, 1 28 2224 51.6 / 52.4; 96 1 32 1523 31.1 / 27.6, but 2 20 1283 27.2 / 28.2; 80 1 26 2246 44.8 / 40.1 (and 5 8 1400
// 30.1 / 28.5, left out with its like); 64 1 24 1466 24.1 / 19.8, 1 40 1461 25.8 / 25.0, 1 44 1350 25.5 / 25.0, but 4 16 854 17.7 /
// 18.5; 32 1 80 582 10.8 / 9.9, 1 96 582 10.95 / 10.90.  Without a mask every walk is as long and halves are slower: 128
// 1 16 2500 64.6 / 77.0.
static bool takes_halves(const FlashTileParams& p, dim3 grid) {
    if (p.pack != 1 || p.decode_rows || p.window != 0 || p.mask == kMaskPadding || p.seq_kv < (p.dim <= 64 ? kHalvesFrom64 : kHalvesFrom)) return false;
    const unsigned long long units = (unsigned long long)grid.x * grid.y, n = units * grid.z, n_cus = (unsigned long long)p.n_cus;
    if (n <= n_cus) return true;
    if (p.mask != kMaskCausal || 10 * n > 19 * n_cus) return false;
    if (p.dim > 64) return grid.z >= 18 || (grid.z >= 11 && units % 8 == 0 && 8 * units <= n_cus && 4 * n <= 7 * n_cus);
    return grid.z >= (p.dim <= 32 ? 5 : 11);
}
// Head dims above 128: the pipelined walk over tiles of 64 keys straight to LDS, one workgroup a CU, or the walk over tiles of 32 through registers,
// whose phases follow one another (one wave a SIMD as well: O takes 128 registers).  us, registers / LDS, B H N at head dim 256 unless it says
// otherwise.  Where the workgroups leave a quarter of the CUs idle or more, the first from 96 keys on: causal 1 8/2 1024 46.5 / 32.7, 2 16 100 11.7 /
// 10.5, 256 16.9 / 13.5, but 1 16 65 9.9 / 10.3, 1 16 16 7.4 / 8.5.  A padded batch of more workgroups than half the CUs, whose lengths are less,
// from 160 (3 28 133 12.6 / 13.6, 2 32 122 at 224 1.06, 4 16 200 1.05 times as fast), a chunk, which requests its first tiles ahead of all else, from
// 140 (16 8 87 positions over 129, head dim 208, 14.9 / 15.8; 11 8 176 over 176, 144, 1.05 times).
// Where they fill the chip the tiles of 64 keys that are asked for ahead of the walk come from memory at the pace of all of them, and a short walk
// ends before they have paid.  Causal 16 16 128 14.7 / 15.9, 32 16 200 61.9 / 65.7, 256 70.1 / 72.8, 300 108.6 / 107.5, 520 228 / 224, 4 32 2048 410
// / 338, head dim 160 32 16 160 45.5 / 48.3, 256 59.4 / 57.7; four query heads a kv head, whose keys the L2s have, 8 32/8 97 12.6 / 12.4, 128 13.7 /
// 14.2 (at 224 1.02 times as fast), 160 24.0 / 23.4, 3 40/8 724 71.7 / 56.7.  None: of 129 to 160 keys, five tiles or three, 32 16 160 55.6 / 57.5,
// else 97 26.3 / 25.5, 200 70.8 / 72.1 (head dim 160 62.1 / 59.2), 256 86.2 / 80.6, 2 16 2048 177 / 130, shared 8 32/8 97 12.9 / 11.5.  A padding
// mask ahead from 97 keys on (32 16 128 34.4 / 31.8, 2 16 2048 202 / 138).  Padded, lengths from a sixth of N: heads that do not divide by the XCDs
// 40 12 260 57.4 / 62.4, 400 86.6 / 90.4, 600 131.9 / 129.1, others 23 16 246 41.0 / 40.7, 27 8 370 42.9 / 40.4, 9 32 1483 266 / 237, head dim 160 16
// 16 320 33.5 / 34.0, 600 70.1 / 64.5.  Windows, of which a workgroup walks a few tiles whatever N is: with keys of their own a window of 130, 8 16
// 3594 at head dim 224 316 / 367, of 228, 5 12 2530 at 208 136 / 143, of 434, 5 16 1424 at 240 119 / 124, at 256 157, 4 32 1357 123 / 134, 278, 6 12
// 2854 183 / 179; shared by two heads an XCD or more 476, 4 40/8 2653 427 / 353, 102, 3 40/8 1562 127 / 112, by one 131, 36 8/2 1186 at 240 256 /
// 278.
// A chunk: 32 16 100 positions over 500 63.5 / 66.3, 1000 118 / 111, 64 32/8 4 over 500 57.1 / 61.0, 2000 181 / 184, 32 8 30 at head dim 224 over
// 1000 46.7 / 48.0, 192 over 400 23.1 / 23.9, 700 34.0 / 32.0, 160 32 16 100 over 200 33.0 / 35.7, 300 40.6 / 39.2, 64 32/8 4 over 300 39.3 / 35.9;
// more than 64 rows of shared kv heads, or a workgroup for each CU at most, times as fast, 6 28/4 219 at 240 over 219 0.98, 15 8 219 over 969 1.12,
// 21 32/8 71 over 288 1.05, 3 32/8 336 at 240 over 782 1.27. Over 1040 drawn calls that fill the chip three of the 587 that the rule sends straight
// to LDS are more than 2 % slower (3.9, 3.3, 2.1), and the mean gain of the 587 is 1.14.
// Spans of a chunk: from 256 keys a span and 97 rows on, 65 of shared kv heads: 1 16/2 100 over 2048 29.1 / 26.1, of 72 rows 11 32/8 18 over 6304 138
// / 130, of 87 1 32 87 over 2812 30.1 / 31.8, of 64 1 32/8 16 over 8192 22.2 / 22.5, of 32 keys 10.2 / 11.4.  Not with a bias, whose LDS leaves the
// query rows to be read into the operands and whose values spill: 4 8 1024 57.2 / 65.0, 1 8 77 x 513 38.6 / 52.1.
// A chunk whose lengths are on the device is taken to be as long as its new positions, from 256 of them on, not as the cache: a length that the
// launch does not know may be short.  max_seq 8192, all lengths alike, at 20, 100, 300, 1000 and 8000 keys: 32 32/8 16 positions 9.8 / 14.5, 14.8 /
// 15.5, 26.0 / 26.2, 60.7 / 60.4, 384 / 378; 9 8 8 10.3 / 12.2, 11.4 / 11.7, 13.7 / 14.5, 23.3 / 25.7, 112 / 112; 32 16 100 - , 29.8 / 33.9, 48.8 /
// 51.1, 119 / 117, 827 / 746; 4 16/2 200 - , - , 30.1 / 30.3, 42.3 / 38.5, 172 / 122; 5 28 96 at 96 and 4000 11.8 / 13.4, 164 / 150; 4 16 300 at 300,
// 1000 and 8000 19.5 / 17.6, 46.4 / 39.2, 319 / 248; 2 16/8 1024 at 1024 and 8000 49.1 / 41.5, 321 / 247. (A padded batch is as long as its longest
// sequence: 5 8 of 2817, lengths 352 to 2817 119 / 97, one of 2817 and the rest 20 116 / 87; all 20, which nobody pads so far, 16.7 / 17.7.)
static bool takes_tiles_direct(const FlashTileParams& p) { return flash_tile_bf16_direct(p); }
template <int DP>
hipError_t launch_dp(hipStream_t stream, const FlashTileParams& p, dim3 grid) {
    if (p.mask == kMaskPadding) {
        // Tiles straight to LDS and a bit per key, as far as the bits fit a stage (from 32768 keys at DP 32 to 131072 at 128).  us,
        // a byte a lane with tiles through registers -> this, the last eighth of the keys hidden, B H N head dim: 2 12 2032 128
        // 72.7 -> 60.7 (no mask 57.0), 1 12 1866 96 43.6 -> 35.9, 3 16 1117 80 33.9 -> 29.5, 4 16 2048 64 87.5 -> 80.3, 8 16 512 64 15.6 ->
        // 14.3, 2 16 3000 32 64.3 -> 63.5.  A single tile at head dim 128 stays: 5 16 42 128 6.2, 6.4.
        if (p.seq_kv <= 8 * TileCfg<DP>::STAGE_BYTES && (DP < 128 || (DP == 128 ? p.seq_kv > TileCfg<DP>::KT : takes_tiles_direct(p)))) {
            if (p.dim == DP) return launch_one<DP, kMaskPadding, false, false, false, false, kTilesDirect>(stream, p, grid);
            return launch_one<DP, kMaskPadding, false, false, false, false, kTilesDirectPart>(stream, p, grid);
        }
        return launch_one<DP, kMaskPadding, false, false>(stream, p, grid);
    }
    if constexpr (DP <= 128) {
        constexpr int kTiles = DP % 64 == 0 ? kTilesDirect : kTilesDirectPart;
        if ((kTiles == kTilesDirectPart || p.dim == DP) && takes_halves(p, grid)) return launch_halves<DP, kTiles>(stream, p, grid);
    }
    if constexpr (DP > 128) {
        if (!takes_tiles_direct(p)) return launch_tiles<DP, kTilesRegs>(stream, p, grid);
    }
    return p.dim == DP ? launch_tiles<DP, kTilesDirect>(stream, p, grid) : launch_tiles<DP, kTilesDirectPart>(stream, p, grid);
}

}  // namespace

bool flash_tile_bf16_supported(int dim) { return dim > 0 && dim <= 256 && dim % 8 == 0; }
static_assert(flash_tile_bf16_key_tile(128, false) == TileCfg<128, true>::KT && flash_tile_bf16_key_tile(136, false) == TileCfg<256>::KT &&
                  flash_tile_bf16_key_tile(136, true) == TileCfg<256, true>::KT,
              "the host's rule of the key tile");
static_assert(flash_tile_bf16_workgroups(64) == TileCfg<64>::OCC && flash_tile_bf16_workgroups(72) == TileCfg<96>::OCC && flash_tile_bf16_workgroups(136) == TileCfg<256>::OCC,
              "the host's rule of the workgroups a CU");
// The kernel addresses the keys of one (batch, kv head) with 32-bit byte offsets (tile offset + lane offset, the
// requests that run a few tiles past the last one included).
bool flash_tile_bf16_addressable(long long seq_kv, long long row_pitch) {
    return seq_kv >= 0 && row_pitch > 0 && (unsigned long long)(seq_kv + 512) * (unsigned long long)row_pitch * 2ull < (1ull << 32);
}

// What the kernels take grid positions for heads by.
static void set_grid_order(FlashTileParams& p, long long z) {
    p.n_qtiles = (int)z;
    p.kv_magic = 0;
    if (p.pack > 1 || p.decode_rows || p.group == 1) return;
    if (p.kv_heads == 1) {  // (2^32 / 1 does not fit the multiplier) every head with keys of its own, at the same address
        p.kv_heads = p.heads;
        p.group = 1;
        p.lkv.head_stride = 0;
        return;
    }
    p.kv_magic = (uint32_t)(0x100000000ull / (unsigned long long)p.kv_heads) + 1u;
}

// 64 rows per wave: head dim 64 exactly, rows of one head, masks none / causal (with or without per-sequence lengths)
bool flash_wide_bf16_supported(const FlashTileParams& p) {
    return p.dim == 64 && p.pack <= 1 && !p.bias && p.n_splits <= 1 && (p.mask == kMaskNone || p.mask == kMaskCausal) &&
           flash_tile_bf16_addressable(p.seq_kv, p.lkv.row_pitch);
}

hipError_t launch_flash_wide_bf16(hipStream_t stream, const FlashTileParams& params) {
    FlashTileParams p = params;
    if (p.batch == 0 || p.heads == 0 || p.seq_q == 0) return hipSuccess;
    if (!flash_wide_bf16_supported(p) || p.group < 1) return hipErrorInvalidValue;
    const long long n_qtiles = ((long long)p.seq_q + WROWS - 1) / WROWS;
    if (p.batch > 65535 || n_qtiles > 65535 || p.heads > 65535) return hipErrorInvalidValue;  // grid limits
    p.pack = 1;
    set_grid_order(p, n_qtiles);
    dim3 grid((unsigned)p.heads, (unsigned)p.batch, (unsigned)n_qtiles);
    if (p.mask == kMaskCausal) hipLaunchKernelGGL(flash_wide_bf16_kernel<kMaskCausal>, grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(flash_wide_bf16_kernel<kMaskNone>, grid, dim3(256), 0, stream, p);
    return hipGetLastError();
}

// A padded batch's query tiles in one order over all sequences (at most 64: a lane each): where they do not fit the chip at
// once, and the walks are long enough to pay for the wait for the lengths ahead of the first request for keys.  us, by
// sequence / by length (with the binary search), inputs that change from pass to pass, lengths spread evenly up to N and
// standing in any order in the batch, B H N shortest head dim: 16 16 1024 170 64 34.5 / 32.8 (33.5), 32 8 2000 333 64 90.2 / 85.0
// (86.3), 20 8 3000 500 128 210 / 193 (193), 4 16 4000 666 128 142.3 / 128.4 (127.2), 22 40 949 158 64 103.5 / 93.9 (97.0), 2 16
// 4000 666 64 61.0 / 53.4 (53.8), 12 16 2048 1024 64 90.6 / 89.2 (91.2).  What the order gains depends on where the long
// sequences stand and how far the lengths lie apart; what is left otherwise is the wait: 3 16 3107 517 64 51.4 / 53.0 (53.4),
// 14 8 1174 195 64 23.9 / 24.5 (25.1), 3 32 1702 283 256 124.2 / 130.6 (130.7), and lengths all equal 16 16 1024 64 55.1 / 55.9
// (56.6), 22 40 949 64 184 / 188 (191), 14 8 1174 64 34.4 / 36.1 (37.3).  With fewer than eight tiles (with the search) 64 8 500
// 64 96 34.7 / 34.6, 12 16 700 100 32 11.9 / 12.6, 22 16 300 60 80 16.3 / 18.6.
static bool tiles_by_length(const FlashTileParams& p, long long n_qtiles) {
    return p.q_lens && p.kv_lens == p.q_lens && p.seq_q == p.seq_kv && p.mask == kMaskCausal && p.pack == 1 && !p.decode_rows && p.window == 0 &&
           p.batch > 1 && p.batch <= 64 && n_qtiles >= 8 &&
           n_qtiles * p.batch * p.heads > (long long)p.n_cus * flash_tile_bf16_workgroups(p.dim);
}

hipError_t launch_flash_tile_bf16(hipStream_t stream, const FlashTileParams& params) {
    FlashTileParams p = params;
    if (p.batch == 0 || p.heads == 0 || p.seq_q == 0) return hipSuccess;
    if (!flash_tile_bf16_supported(p.dim) || p.pack < 1) return hipErrorInvalidValue;
    if (p.bias && (p.mask != kMaskNone || !flash_tile_bf16_bias_addressable(p.seq_kv))) return hipErrorInvalidValue;
    if (!flash_tile_bf16_addressable(p.seq_kv, p.lkv.row_pitch)) return hipErrorInvalidValue;
    if ((p.pack > 1 || p.decode_rows) && (p.bias || p.mask != kMaskCausal)) return hipErrorInvalidValue;  // packed rows: the chunked decode only
    if (p.window < 0 || (p.window > 0 && (p.pack > 1 || p.decode_rows || p.bias || p.mask != kMaskCausal || p.n_splits > 1))) return hipErrorInvalidValue;
    const long long rows = (long long)p.seq_q * p.pack;
    const long long n_qtiles = (rows + TROWS - 1) / TROWS;
    const long long heads_u = (p.pack > 1 || p.decode_rows) ? p.kv_heads : p.heads;
    if (p.n_splits < 1) p.n_splits = 1;
    if (p.n_splits > 1 && (p.pack != p.group || p.bias || p.mask != kMaskCausal || !p.part_o || !p.part_ml))
        return hipErrorInvalidValue;  // the chunked decode only
    // (what is cut leaves CUs idle: fewer than 2^15 rows and slabs.  The merge's grid, its offsets and its divisions need no more.)
    if (p.n_splits > 1 && ((long long)p.batch * p.kv_heads > 65535 || (rows + 31) / 32 > 65535 || rows * (long long)p.pack >= 1ll << 32 ||
                           (long long)p.batch * p.kv_heads * p.kv_heads >= 1ll << 32 || (long long)p.n_splits * p.dim >= 1ll << 25))
        return hipErrorInvalidValue;
    if (p.batch > 65535 || n_qtiles * p.n_splits > 65535 || heads_u > 65535 || p.group < 1) return hipErrorInvalidValue;  // grid limits
    set_grid_order(p, n_qtiles * p.n_splits);
    if (tiles_by_length(p, n_qtiles)) p.n_qtiles = -1;
    dim3 grid((unsigned)heads_u, (unsigned)p.batch, (unsigned)(n_qtiles * p.n_splits));
    if (p.dim <= 32) return launch_dp<32>(stream, p, grid);
    if (p.dim <= 64) return launch_dp<64>(stream, p, grid);
    if (p.dim <= 96) return launch_dp<96>(stream, p, grid);
    if (p.dim <= 128) return launch_dp<128>(stream, p, grid);
    return launch_dp<256>(stream, p, grid);
}

}  // namespace rt
