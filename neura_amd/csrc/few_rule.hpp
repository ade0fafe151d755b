// Which wide products are the product of few rows' (gemm_few.hip) and which the 128 x 128 tiles' (gemm.hip), and which narrow products
// go there: plain C++, so that the rules can be held to the measured points without a device.
#pragma once
#include "../../include/neura_hip.h"

#include <cstdint>

namespace nh {

// Tiles of 32 packed rows a wave multiplies its unpacked weights by: one, or two or three -- passes over the weights, each the time of
// its row tiles and of one more for the weights.  A matrix whose 32-column tiles leave half of the compute units without one is bound by
// how much is in flight and takes twos (attn_output of the 7B shape: 48 rows in threes 18.6 us, 64 rows in twos 16.7; gate: 22.4, 26.0).
inline uint32_t few_row_tiles(uint32_t N, uint32_t rows, uint32_t compute_units) {
    const uint32_t row_tiles = (rows + 31u) / 32u, tiles = (N + 31u) / 32u;
    if (row_tiles <= 1u) return 1u;
    if (tiles <= compute_units / 2u) return 2u;
    return (row_tiles + 1u) / 2u * 3u <= (row_tiles + 2u) / 3u * 4u ? 2u : 3u;
}

// Where the line lies.  Up to 96 packed rows most of a tile of 128 is padding (7B shape, Q4_K, 16 rows of fp32: gate|up 74 -> 36 us).
// Past that the tiles take whole rounds of one workgroup a compute unit, however few of them the last round has, and the product
// of few rows takes the time of its work: `share` hundredths of what a tile costs, by format and by the row tiles a pass over the
// weights serves.  A round costs the tiles 350 k more than it walks (filling and draining).  Shares are fitted to both forms timed at
// 128 to 8192 packed rows over the 0.5B, 1.5B and 7B shapes (us, tiles / few): Q8_0 18944 x 3584 at 512 rows 157 / 211 and at 1024 262 /
// 331 (full rounds), 3584 x 3584 at 512 56 / 48 (112 workgroups), 4608 x 3584 at 1024 105 / 87 (288), 4864 x 896 at 1024 47 / 35 (304);
// Q6_K 221 / 193, 80 / 47, 151 / 96 of the first, third and fourth; Q3_K 155 / 140, 57 / 39, 107 / 71; Q5_K 141 / 150, 51 / 40, 95 / 76; Q4_K
// 125 / 148, 43 / 39, 82 / 77.  The form it picks is within 8 % of the faster one at those points.
inline bool few_rows_win(int32_t element, uint32_t N, uint32_t K, uint32_t rows, uint32_t compute_units) {
    if (rows <= 96u) return true;
    if (rows > 65535u * 32u) return false;  // (row tiles are blockIdx.y)
    struct Share {
        uint32_t twos, threes;
    };
    const Share share = element == NH_Q8_0   ? Share{195u, 145u}
                        : element == NH_Q6_K ? Share{105u, 95u}
                        : element == NH_Q5_K ? Share{180u, 140u}
                        : element == NH_Q3_K ? Share{120u, 109u}
                                             : Share{200u, 170u};
    const uint64_t groups = (uint64_t)((N + 127u) / 128u) * ((rows + 127u) / 128u), rounds = (groups + compute_units - 1u) / compute_units;
    const uint64_t tiles_cost = 100u * rounds * compute_units + (rounds - 1u) * compute_units * 35000u / K;
    return groups * (few_row_tiles(N, rows, compute_units) == 3u ? share.threes : share.twos) <= tiles_cost;
}

// The same for two to eight rows of a narrow product, against the vector and staged kernels (gemv.hip), which walk the weights once for
// every four, two or one rows.  Q4_K has tiles of its own and stays (7B shape, eight rows: gate|up 26 against 36 us, ffn_down 23 against
// 27).  Of the others three rows and five are two passes or more and go (7B shape, eight rows: Q8_0 gate|up 304 -> 62, Q6_K ffn_down 101 ->
// 34; the worst of 53 shapes at three rows: 1.06 times).  Two and four rows are one pass.  The staged kernel takes eight columns and a
// slice of K a workgroup: up to two workgroups a compute unit it is one round of latency, which the packing launch alone does not
// beat (4096 x 3584, 512 of them, two rows: Q3_K 8.9 against 11.7, Q5_K 10.2 against 12.4, Q6_K 9.8 against 15.3), and a second
// round costs more than all of the product here (4608 x 3584, 576: Q3_K 14.3 -> 11.9, Q5_K 16.4 -> 12.5; four rows of 3584 x 3584, 896:
// Q3_K 18.3 -> 12.2, Q6_K 18.4 -> 15.8).  Four rows of Q5_K fill a compute unit's LDS with one (2048 x 1536, 256: 8.0 against 8.7; 3584 x
// 3584 27 -> 13).  Two gated rows of Q6_K, two planes of MFMAs over two matrices, are worth it later (17920 x 1536 20.3 against 21.3,
// 37888 x 3584 57 -> 52).  Q8_0 streams on the vector kernel without rounds; two rows of it go where the walk outweighs the packing, 46 K
// numbers a compute unit (3584 x 3584 18.5 -> 13.5, 2688 x 4096 13.0 against 15.1).  Over 1245 products timed in both forms the pick takes
// 1.003 times the faster one's time on average.
inline bool few_narrow_rows_win(int32_t element, uint32_t N, uint32_t K, uint32_t rows, bool gated, uint32_t compute_units) {
    if (element == NH_Q4_K) return false;
    if (rows == 3u || rows >= 5u) return true;
    if (element == NH_Q8_0) return rows == 4u || (uint64_t)N * K >= 46000u * (uint64_t)compute_units;
    const uint64_t blocks = K / 256u, most = rows == 4u ? 8u : 16u, workgroups = (N + 7u) / 8u * ((blocks + most - 1u) / most);
    if (element == NH_Q5_K && rows == 4u) return workgroups > compute_units;
    if (element == NH_Q6_K && rows == 2u && gated) return workgroups > 12u * (uint64_t)compute_units;
    return workgroups > 2u * (uint64_t)compute_units;
}

}  // namespace nh
