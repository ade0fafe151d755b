// How the Q4_K product of several activation rows (gemv_rows.hip) is dealt, what its plans take of LDS and of scratch: plain C++, so that every
// plan can be checked without a device.
#pragma once
#include <cstddef>
#include <cstdint>

namespace nh {

constexpr uint32_t ROWS_MOST_BLOCKS = 16, ROWS_MOST_BLOCKS_MANY = 7;  // super-blocks of a slice: up to eight rows, and nine to sixteen

// Bytes of LDS a staged super-block takes: a row tile's operands, [MFMA][kq] of sixteen 16-byte pieces, row r of lane group kq in place r ^ kq
// and 64 bytes of padding behind an MFMA's 1 KB (the sixteen lanes that stage a row write to different banks, and an operand is
// still 1 KB in a row); its sub-blocks' sums in fp32, [h][kq] of sixteen A rows: of sub-block 4 (kq & 1) + 2 (kq / 2) + h; the rows' scales.
constexpr uint32_t ROWS_OPERAND = 1024u + 64u, ROWS_SUMS = 8u * ROWS_OPERAND, ROWS_TILE = ROWS_SUMS + 8u * 64u, ROWS_SCALES = 8u * 4u;
constexpr uint32_t rows_block_bytes(uint32_t rt) { return rt * (ROWS_TILE + ROWS_SCALES); }
constexpr size_t rows_lds(uint32_t blocks, uint32_t rt, uint32_t waves, uint32_t shares) {
    return (size_t)blocks * rows_block_bytes(rt) + (size_t)8u * rt * ROWS_MOST_BLOCKS * 4u + (shares > 1u ? (size_t)waves * rt * 1024u : 0u);
}
// passes of a workgroup over the rows it stages, sixteen lanes a super-block, and the rows of one pass where a slice has `blocks` of them
constexpr uint32_t rows_passes(uint32_t waves) { return (32u + waves - 1u) / waves; }
constexpr uint32_t rows_seats(uint32_t blocks) { return blocks <= 4u ? 2u : blocks <= 8u ? 3u : 4u; }  // (a power of two of super-blocks)
constexpr uint32_t rows_hop(uint32_t waves, uint32_t blocks) { return (4u * waves) >> rows_seats(blocks); }

// How a product is dealt: waves a workgroup, how many of them share a tile's super-blocks, and K slices.
struct RowsPlan {
    uint32_t waves, shares, splits;
};

// Up to sixteen super-blocks a row are one slice (LDS: 148 KB of operands at sixteen, 4 to 14 of the waves' sums), deeper ones slices of at most
// fourteen, which a fold adds up.  From four tiles a compute unit on waves walk several super-blocks of several tiles; below, a workgroup
// takes a tile or two and every wave a super-block or three.  With a tile a compute unit at most, a workgroup of one tile: a second slot's waves
// would only stage (us, three and eight rows, 12 or 16 waves / 8: 3584 x 3584 6.9 and 8.0 / 5.6 and 7.4, 2560 x 2048 7.2 and 7.4 / 5.3 and 5.9, 1536 x
// 1536 5.8 and 6.1 / 4.8 and 5.5; 4608 x 3584, a second round for 32 of them, 7.0 and 8.2 / 7.2 and 9.1).
// Eight rows, us (the forms before / 14 waves of 7 shares, 10 of 2, 12 of 6, 16 of 8): gate|up of the 7B shape 28.2 / 22.2, 24.1, -, -; the head
// 77 / 67; q|k|v 10.4 / 9.3, -, 9.1, 9.4; ffn_down 21.8 / 18.4, 25, 18.7, 18.7; of the 1.5B shape, six super-blocks a row, gate|up 14.2 / -, 9.1, 10.1,
// 11.5; ffn_down 12.1 / 11.7, -, -, 11.4.
// Rows of 4096 numbers, three and eight of them (the forms before / slices of eight super-blocks and their fold / one slice): 4096 x 4096 8.4 and 21.3 / 10.4
// and 10.6 / 5.6 and 7.5, 6144 10.5 and 25.8 / 10.6 and 11.2 / 7.8 and 10.0, gate|up of 28672 24.3 and 25.5 / 21.8 and 22.4 / 19.7 and 21.3.
// Precision, 2-norm from 64 bits at eight rows (1e-7; the integer tiles before / minimums and codes weighed apart, sums as halves / here): N(0, 1) rows,
// attn_output 1.91 / 1.34 / 1.24, gate 2.27 / 2.27 / 1.25, ffn_down 1.81 / 1.42 / 1.35; rows of mean 1, 4.84 / 5.43 / 1.66, 17.2 / 17.4 / 1.65, 4.62 / 5.45 /
// 1.71; three rows of attn_output 3.16 / 1.32 / 1.26 and 11.9 / 5.43 / 1.66.  Without any minimum codes are not centred (an outlier at a weight
// of zero leaves its neighbours alone) and add up over a super-block, not a sub-block: 1.05 / 1.27 / 1.27.  It costs the tall ones
// 0.9 us of 21 (the fp32 MFMAs: 32 clocks each on matrix cores busy 15 % of a time that the vector unit fills for 61 %), and the others gain.
// Nine to sixteen rows (`many`) take seven super-blocks a slice, what LDS holds of both their sets: packing and product of few rows there /
// here at sixteen rows of the 1.5B shape: gate|up 19.8 / 13.5, q|k|v and its rotation 13.6 / 11.7, attn_output 10.5 / 9.6, ffn_down 16.6 / 14.3.
// (By shape alone: a product gives the same numbers with the rotation in it and without, whichever planes are active.)
constexpr uint32_t ROWS_SHORT = 256, ROWS_TALL = 1024;  // tiles, one and four for each of 256 compute units
inline RowsPlan rows_plan(uint32_t tiles, uint32_t nblk, bool many) {
    const uint32_t most = many ? ROWS_MOST_BLOCKS_MANY : nblk <= ROWS_MOST_BLOCKS ? ROWS_MOST_BLOCKS : 14u;
    uint32_t splits = (nblk + most - 1u) / most;
    const uint32_t blocks = (nblk + splits - 1u) / splits;
    splits = (nblk + blocks - 1u) / blocks;
    if (tiles * splits >= ROWS_TALL) return blocks > 8u ? RowsPlan{14u, 7u, splits} : RowsPlan{10u, 2u, splits};
    if (!many && (blocks > 14u || tiles * splits <= ROWS_SHORT)) return RowsPlan{8u, 8u, splits};
    return blocks > 8u ? RowsPlan{12u, 6u, splits} : RowsPlan{16u, 8u, splits};
}

// the slices' sums, and of each its rows' sums of squares
inline size_t rows_scratch_bytes(uint32_t N, uint32_t K, uint32_t rows) {
    const uint32_t splits = rows_plan(N / 16u, K / 256u, rows > 8u).splits;
    return splits > 1u ? (size_t)splits * rows * (N + 1u) * sizeof(float) : 0u;
}

}  // namespace nh
