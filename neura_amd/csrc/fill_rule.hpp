// How many workgroups share the walk of a fill's attention (attention.hip): plain C++, so that the rule can be held to the measured
// points without a device.
#pragma once
#include <cstdint>

namespace nh {

constexpr uint32_t FILL_SECTIONS_MOST = 32;

// How many workgroups share the walk of a block of query rows in a fill.  A block's walk is a chain of rounds (a tile a set of waves)
// behind queries, first tile and meeting; blocks times sections come in turns of the chip; sections leave their sums in memory for a
// fold of 4 us and more (480 rows of 28 heads in two: 10 us).  In hundredths of a microsecond, for what the block walks with:
//   halves, two sets of waves   a round of 64 keys 2.35 us at width 128, 1.85 at 64, behind 10 (6.5); one workgroup a compute unit.
//       Over 40 shapes of 5 to 480 rows behind 0 to 1500 kept positions the pick takes 1.005 times the best one's time; 28 heads of 128,
//       one workgroup a block -> here: 37 rows behind 700 41 -> 18 us, 100 behind 1500 72 -> 29, 480 behind 700 59 -> 49; 480 alone stay (31).
//   halves, one set (windows below four tiles)   a round of 32 keys 1.3 (1.0) us behind 4: over 24 shapes 1.006 times the best one's time;
//       with the line above some took 8 % more than walked whole (14 heads of 64, 37 rows behind 60, four planes: 11.8 -> 12.8 us).
//   single states   a round of 32 keys 3.0 (2.0) us behind 4; two workgroups share a compute unit, and each walks 1.6 times as long then.
//       Over 52 shapes 1.001 times the best one's time, 1.04 at most; one workgroup a block -> here, width 128: 37 rows behind 700 73 ->
//       21 us, four planes of 100 behind 1500 156 -> 77 (with the first line 99), 480 behind 700 115 -> 65 (78).
inline uint32_t fill_sections(uint32_t blocks, uint32_t rounds, uint64_t numbers, uint32_t width, bool single, bool split, uint32_t compute_units) {
    const uint32_t round = single ? (width > 64u ? 300u : 200u) : split ? (width > 64u ? 235u : 185u) : width > 64u ? 130u : 100u;
    const uint32_t base = single || !split ? 400u : width > 64u ? 1000u : 650u, slots = single ? 2u * compute_units : compute_units;
    uint32_t best = 1;
    uint64_t least = UINT64_MAX;
    for (uint32_t s = 1; s <= FILL_SECTIONS_MOST && s <= rounds; s++) {
        const uint64_t workgroups = (uint64_t)blocks * s, turns = (workgroups + slots - 1u) / slots;
        const uint64_t walk = (uint64_t)((rounds + s - 1u) / s) * (workgroups > compute_units && single ? round * 8u / 5u : round) + base;
        const uint64_t cost = turns * walk + (s > 1u ? 400u + numbers / 3500u + numbers * s / 7500u : 0u);
        if (cost < least) least = cost, best = s;
    }
    return best;
}

}  // namespace nh
