// Where the bf16 tile kernel keeps what lies in LDS when its tiles travel straight there: plain
// arithmetic, so that a host test can hold every wave's writes against each other.
//
//   [K stage 0][K stage 1][V stage 0][V stage 1]   a stage: KT rows of DP columns without padding
//                                    [query rows ]  128 rows, two stages long, until the first barrier
//                                           [keep]  a bit per key under a key-padding vector, behind that barrier
//
// A wave's load instruction fills 1 KB with 64 chunks of 16 bytes, lane l the 16 bytes at 16 l; instruction n of wave w fills
// block w + 4 n of a stage: chunk 64 (w + 4 n) + l, which is slot chunk % SPR of row chunk / SPR.  Bank conflicts are avoided by
// an XOR of the slot index with bits of the row (K and query rows are read 16 at a time at one slot, V rows 4 at a time over 4
// adjacent slots by the transposing reads; four rows of 64 or of 192 bytes start at four different quarters of the banks,
// which is all that V asks for), applied on the way in: the lane fetches the columns that belong at its LDS position.
#pragma once

namespace rt {

template <int DP>
struct TileLds {
    static constexpr int KT = 64;      // keys per tile
    static constexpr int SPR = DP / 8;  // 16-byte slots per row
    static constexpr int ROW_BYTES = 2 * DP, STAGE_BYTES = KT * ROW_BYTES;
    static constexpr int REQUESTS = KT * SPR / 256;  // load instructions per wave, matrix and tile
    static constexpr int K_AT = 0, V_AT = 2 * STAGE_BYTES, Q_AT = 3 * STAGE_BYTES, KEEP_AT = 4 * STAGE_BYTES;
    static constexpr int Q_REQUESTS = SPR / 2;  // per wave, of its own 32 query rows

    static constexpr int swz_k(int row) { return DP >= 128 ? (row & 15) : (DP == 64 ? ((row >> 1) & 7) : ((row >> 2) & 3)); }
    static constexpr int swz_v(int row) { return DP >= 128 ? 4 * (row & 3) : (DP == 64 ? 4 * ((row >> 1) & 1) : 0); }
    // Instructions n and n + SETS of a wave fetch the same columns, rows_on(n + SETS) - rows_on(n) rows apart: the lane's part of
    // the address is that of instruction n % SETS (whose own rows it holds).
    static constexpr int SETS = DP == 96 ? REQUESTS : (DP == 256 ? 2 : 1);
    static constexpr int rows_on(int n) { return (n - n % SETS) * 256 / SPR; }

    static constexpr int block(int wave, int n) { return 1024 * (wave + 4 * n); }                      // within a stage
    static constexpr int q_block(int wave, int n) { return Q_AT + wave * 32 * ROW_BYTES + 1024 * n; }

    // Head dims between the tile widths: the columns behind the head dim are not requested.  Those of the first CLEARED
    // stages, K's, are zeros from the start: they meet the queries' zeros in the score product, and what an earlier workgroup
    // left there may be infinite or NaN.  V's hold what is there: a column of V makes the same column of O, and those behind
    // the head dim are never stored.  No wave may clear what lies behind V stage 0 either: the query rows of other waves land
    // there, and the first barrier comes behind both.
    static constexpr int CLEARED = 2;
};

}  // namespace rt
