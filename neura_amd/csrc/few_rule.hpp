// Which wide products are the product of few rows' (gemm_few.hip), which the product of shared rows' (gemm_wide.hip) and which the
// 128 x 128 tiles' (gemm.hip), and which narrow products go to the first: plain C++, so that the rules can be held to the measured points without a device.
#pragma once
#include "../../include/neura_hip.h"

#include <cstdint>
#include <initializer_list>

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
// Q5_K 141 / 150, 51 / 40, 95 / 76 of the first, third and fourth; Q4_K 125 / 148, 43 / 39, 82 / 77.  The form it picks is within 8 % of the
// faster one at those points.  (`share` goes by few_row_tiles: threes that few_pass_tiles takes beyond it are at few columns, where the shares of twos
// decide as well; asked for them the rule moves 4 of 1368 points of such matrices, 3 % slower.)  Q6_K and Q3_K have no tiles: few rows up to the height of a grid, and shared rows below.
inline bool few_rows_win(int32_t element, uint32_t N, uint32_t K, uint32_t rows, uint32_t compute_units) {
    if (rows <= 96u) return true;
    if (rows > 65535u * 32u) return false;  // (row tiles are blockIdx.y)
    if (element == NH_Q6_K || element == NH_Q3_K) return true;
    struct Share {
        uint32_t twos, threes;
    };
    const Share share = element == NH_Q8_0 ? Share{195u, 145u} : element == NH_Q5_K ? Share{180u, 140u} : Share{200u, 170u};
    const uint64_t groups = (uint64_t)((N + 127u) / 128u) * ((rows + 127u) / 128u), rounds = (groups + compute_units - 1u) / compute_units;
    const uint64_t tiles_cost = 100u * rounds * compute_units + (rounds - 1u) * compute_units * 35000u / K;
    return groups * (few_row_tiles(N, rows, compute_units) == 3u ? share.threes : share.twos) <= tiles_cost;
}

// How the product of few rows splits the K of a tile of columns: `deep` waves a workgroup, `slices` workgroups; rows in tiles of `mt` a
// pass, `nt` matrices beside each other (gated).  The split that walks the fewest units: rounds of workgroups times the units of a wave
// (and what a workgroup takes before its first and after its last, about two units' time).  A matrix of few tiles and deep rows
// leaves most of the chip idle that way, so K may be shared among workgroups too: their meeting costs a unit's time and the passage of
// their sums, 2.5 MB in another (eight rows of fp32, with the packing: ffn_down of the 7B shape Q8_0 55 -> 37 us, Q6_K
// 45 -> 34, Q5_K 37 -> 29, of the 1.5B shape Q8_0 28 -> 18; gate|up of the 7B shape, 592 tiles, is better left alone: Q4_K 34, not 38).
struct FewSplit {
    uint32_t deep, slices, cost;  // cost in 64ths of a unit
};
constexpr uint32_t FEW_SLICES_MOST = 8, FEW_MEETS_MOST = 1024;
constexpr uint64_t FEW_SUMS_MOST = 16u << 20;  // bytes
inline FewSplit few_split(int32_t element, uint32_t N, uint32_t K, uint32_t rows, uint32_t mt, uint32_t nt, uint32_t compute_units) {
    const uint32_t steps = element == NH_Q8_0 ? 2u : 4u, units = (K / 64u + steps - 1u) / steps, tiles = (N + 31u) / 32u, row_tiles = (rows + 31u) / 32u;
    const uint64_t places = (uint64_t)tiles * ((row_tiles + mt - 1u) / mt);
    FewSplit best = {1u, 1u, ~0u};
    for (uint32_t deep = 1; deep <= 8u; deep++)
        for (uint32_t slices : {1u, 2u, 3u, 4u, 6u, FEW_SLICES_MOST}) {
            const uint32_t resident = compute_units * (8u / deep);
            if (slices > 1u && (places > FEW_MEETS_MOST || deep * slices > units || slices * places * mt * nt * 4096u > FEW_SUMS_MOST)) continue;
            const uint32_t meeting = slices > 1u ? 64u + (uint32_t)((uint64_t)slices * N * nt * rows * 4u * 64u / 2500000u) : 0u;
            const uint32_t cost = (uint32_t)((places * slices + resident - 1u) / resident) * ((units + deep * slices - 1u) / (deep * slices) + 2u) * 64u + meeting + deep;
            if (cost < best.cost) best = FewSplit{deep, slices, cost};
        }
    return best;
}

// The row tiles a pass of the product of few rows takes.  Where few_row_tiles has twos for want of column tiles, threes all the same if their
// passes, split as they are best split, cost less: fewer workgroups, each a longer walk, and where twos start a second round or leave a
// slice to meet, the shorter one (us, twos / threes: 896 x 4864 Q8_0 at 800 packed rows 37.0 / 29.1, at 960 38.0 / 43.5; 3584 x 18944 Q8_0 at 74
// 55.1 / 44.6, Q6_K 53.0 / 46.0, Q4_K 42.2 / 39.3, at 104 43.1 / 54.0; 3584 x 3584 Q6_K at 140 24.4 / 20.2; 1536 x 8960 Q8_0 at 400 47.4 / 39.5).  Over
// 239 products of the decoder shapes at 74 to 960 packed rows it takes 0.975 times the twos' time, at most 1.017; over 1368 of matrices of up to
// 4096 columns at 66 to 1024 the pass it picks takes 1.007 times the faster one's time, with a ratio of each element's own (1.16 to 1.37 for 6 / 5)
// 1.009.  Never with fewer shares of K: those add up less exactly.
inline uint32_t few_pass_tiles(int32_t element, uint32_t N, uint32_t K, uint32_t rows, uint32_t compute_units) {
    const uint32_t mt = few_row_tiles(N, rows, compute_units);
    if (mt != 2u || rows <= 64u || (N + 31u) / 32u > compute_units / 2u) return mt;
    const FewSplit twos = few_split(element, N, K, rows, 2u, 1u, compute_units), threes = few_split(element, N, K, rows, 3u, 1u, compute_units);
    // (a unit of a wave takes its row tiles' time and that of three more for its weights)
    return threes.cost * 6u < twos.cost * 5u && threes.deep * threes.slices >= twos.deep * twos.slices ? 3u : 2u;
}

// units of K: 256 numbers, 128 of Q8_0
inline uint32_t shared_rows_units(int32_t element, uint32_t K) { return element == NH_Q8_0 ? (K / 64u + 1u) / 2u : (K / 64u + 3u) / 4u; }

// Units of k a wave of the product of shared rows adds up before its sums leave the accumulators (a chain): as many as a share of the
// product of few rows has in the passes of few_row_tiles (threes by cost have as many or more), where that is the form it takes over from, for one chain over all of K adds up less exactly than shares that
// meet (2-norm from 64 bits, few rows / one chain / here: Q3_K 3584 x 18944 at 600 packed rows 1.15e-7 / 1.75 / 1.16, Q6_K at 800 1.56 /
// 2.41 / 1.56, Q5_K at 600 1.56 / 1.99 / 1.49, Q8_0 17920 x 1536 at 200 1.10 / 1.38 / 1.10).  The tiles are one chain themselves.
inline uint32_t shared_rows_chain(int32_t element, uint32_t N, uint32_t K, uint32_t rows, uint32_t compute_units) {
    const uint32_t units = shared_rows_units(element, K);
    if (!few_rows_win(element, N, K, rows, compute_units)) return units;
    const FewSplit split = few_split(element, N, K, rows, few_row_tiles(N, rows, compute_units), 1u, compute_units);
    return (units + split.deep * split.slices - 1u) / (split.deep * split.slices);
}
// Sums of chains that registers hold, of a row tile's sixteen a lane: of two tiles all, of three the eight of whole rows (every second row
// holds residues, whose sums run on in one chain), which Q6_K in four waves, two planes of operands, leaves no room for.
constexpr int shared_rows_spare(int32_t element, uint32_t waves, uint32_t mt) { return mt == 2u ? 16 : mt == 3u && !(element == NH_Q6_K && waves == 4u) ? 8 : 0; }
// Beside residuals, whose place is the outputs', the sums of chains wait in scratch: whether they do, and are more than that holds
inline bool shared_rows_overflow(int32_t element, uint32_t N, uint32_t K, uint32_t rows, uint64_t residual_bytes, uint32_t compute_units) {
    return residual_bytes > FEW_SUMS_MOST && shared_rows_chain(element, N, K, rows, compute_units) < shared_rows_units(element, K);
}

// Where the product of shared rows (gemm_wide.hip) takes over, and in which shape: waves side by side and row tiles a wave (none: the form
// that few_rows_win picks).  Times in microseconds of all three, each a line fitted to 649 products of the decoder shapes at 20 to
// 1024 packed rows (mean error 4 % here, 4 % of the tiles, 7 % of the product of few rows): turns of the chip, a base and the units
// (256 k, Q8_0 128) of each; two workgroups of four waves share a compute unit, and one alone walks faster.  It wants to win by
// 8 %, so that no line's error makes a product slower: where it is picked it takes 0.9 of the other form's time on average, at most 1.05
// (7B shape, packed rows, other / here: gate|up Q4_K 74 56 / 50, 128 76 / 65, 400 208 / 188, 1024 406 / 344; Q3_K 1024 436 / 329;
// Q8_0 200 and ffn_down Q4_K 300 tie).  Over 1368 products of matrices of up to 4096 columns at 66 to 1024 packed rows what is picked takes 1.005 times the
// fastest form's time.  The lines are of one matrix again and again, which the Infinity Cache holds; over matrices from
// HBM every form takes 2 to 15 % longer in the same order (gate|up Q4_K 74 63 / 58, 128 82 / 67, 1024 407 / 352).  Up to two row tiles the
// walk is latency, not work.
enum SharedShape { SHARED_NONE = 0, SHARED_42 = 42, SHARED_43 = 43, SHARED_83 = 83, SHARED_84 = 84 };
inline SharedShape shared_rows_shape(int32_t element, uint32_t N, uint32_t K, uint32_t rows, bool halves, uint32_t compute_units) {
    if (rows <= 64u || !N || !K || !compute_units) return SHARED_NONE;
    struct Times {
        double tiles, twos, threes;             // of a 128 x 128 tile's 256 k (Q6_K, Q3_K: none); of a unit of the product of few rows, two or three row tiles a pass
        double pair2, one2, pair3, one3, e3, e4;  // of a unit here: 4 x 2 with company and alone, 4 x 3, 8 x 3, 8 x 4
    };
    const Times t = element == NH_Q8_0   ? Times{2.73, 2.26, 2.63, 1.82, 1.41, 2.21, 1.55, 0.0, 2.74}
                    : element == NH_Q6_K ? Times{0.0, 3.41, 4.68, 4.04, 2.41, 4.90, 2.66, 4.26, 0.0}
                    : element == NH_Q5_K ? Times{2.34, 2.86, 3.74, 2.79, 1.71, 3.36, 1.89, 2.84, 3.28}
                    : element == NH_Q3_K ? Times{0.0, 2.66, 3.38, 2.47, 1.65, 2.96, 1.87, 2.64, 2.90}
                                         : Times{1.69, 2.68, 3.56, 2.44, 1.49, 3.11, 1.72, 2.49, 3.04};
    const uint64_t cu = compute_units, row_tiles = (rows + 31u) / 32u;
    const uint32_t per = element == NH_Q8_0 ? 128u : 256u, units = (K + per - 1u) / per;
    const double millions = (double)rows * K * 1e-6;  // (packed, and read again)
    double other;
    if (few_rows_win(element, N, K, rows, compute_units)) {
        const uint32_t mt = few_pass_tiles(element, N, K, rows, compute_units);  // (the passes that are launched)
        const double walk = few_split(element, N, K, rows, mt, 1u, compute_units).cost / 64.0;
        other = mt == 3u ? 2.2 + t.threes * walk + 5.0 * millions : 3.8 + t.twos * walk + 3.2 * millions;
    } else {
        const double rounds = (double)(((uint64_t)((N + 127u) / 128u) * ((rows + 127u) / 128u) + cu - 1u) / cu);
        other = 3.0 + rounds * (9.5 + t.tiles * K / 256.0) + 3.1 * millions;
    }
    SharedShape best = SHARED_NONE;
    double least = other / 1.08;
    // Places between chains, and the end: nothing where three row tiles keep whole rows' sums in registers, 2 microseconds a turn for two
    // (which leave a compute unit two workgroups in place of three: 18944 x 3584 Q3_K at 400 packed rows 108 -> 120) and through memory (84:
    // 37888 x 3584 Q3_K at 200 130.0 -> 137.1), 7 of half rows there, which have twice the sums.
    // `halves`: rows of half activations.  Their outputs are twice as many too, 2 us here and not in few rows, whose shares meet
    // in LDS: over 400 products of 70 to 1024 of them the pick takes 1.003 times the fastest form's time, at most 1.01 times the other
    // form's; with the line of whole rows up to 1.26 (17920 x 1536 at 200 Q3_K few rows 32.9, 83 41.4).
    const uint32_t chain = shared_rows_chain(element, N, K, rows, compute_units), places = chain < units ? (units - 1u) / chain + 1u : 0u;
    const auto consider = [&](SharedShape shape, uint32_t waves, uint32_t mt, double pair, double one, double base, double turn, double pack) {
        if (!(pair > 0.0)) return;
        const uint64_t workgroups = (uint64_t)((N + 32u * waves - 1u) / (32u * waves)) * ((row_tiles + mt - 1u) / mt), slots = waves == 4u ? 2u * cu : cu;
        const uint64_t full = workgroups / slots, left = workgroups % slots;
        const bool lone = waves == 4u && left && left <= cu;
        const uint64_t turns = full + (left ? 1u : 0u);
        const double place = mt == 2u ? 2.0 : halves ? 7.0 : shared_rows_spare(element, waves, mt) ? 0.0 : 2.0;
        const double time = base + (halves ? 2.0 : 0.0) + (double)turns * (turn + units * pair + place * places) - (lone ? units * (pair - one) : 0.0) + pack * millions;
        if (time < least) least = time, best = shape;
    };
    consider(SHARED_42, 4u, 2u, t.pair2, t.one2, 5.0, 5.5, 1.7);
    consider(SHARED_43, 4u, 3u, t.pair3, t.one3, 2.0, 12.0, 1.5);
    consider(SHARED_83, 8u, 3u, t.e3, t.e3, 1.0, 14.5, 1.4);
    consider(SHARED_84, 8u, 4u, t.e4, t.e4, 0.0, 18.0, 1.2);
    return best;
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
