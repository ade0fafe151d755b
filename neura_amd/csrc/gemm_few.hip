// The wide product of few activation rows: Y[m][n] = sum_k X[m][k] * W[n][k] where 128 x 128 tiles (gemm.hip) would be a few dozen
// workgroups (a chunk of a short prompt, a step of more planes than the narrow products take).
//
// What bounds it is weight bytes in flight: a wave walks weight rows of 32 columns, a super-block of k at a time, the next
// super-block's blocks on their way while it unpacks and multiplies this one's.  A workgroup is up to eight waves over one tile of
// columns that share K (wave `share` takes super-blocks share, share + deep, ...); they meet once, in LDS, at the end of the walk, so
// nothing in the walk waits for another wave.  Where a matrix has too few column tiles for the chip, `slices` workgroups share the K
// of a tile as well: each leaves its sums in memory (`partial`, past the caches that workgroups do not share) and counts itself in
// the tile's word of `meets`; the last to arrive adds them in the order of the slices and sets the word back to zero.  That
// rests on the launches of a device following each other on its one stream and on the words being zero between them.
//
// v_mfma_f32_32x32x16_f16: the weights are B (lane l32 + 32 part unpacks the numbers of ITS column in registers: runs of 16
// stored numbers at 32 i + 16 part, which for every format are the pieces its blocks are stored in), the packed activation rows
// are A, read in operand order (few_operand_at: 1 KB in a row a wave) a whole step of 64 k ahead or more.  The arithmetic is that
// of the 128 x 128 kernels: exact half operands code * sub-scale, fp32 sums weighed by d a super-block (Q8_0: a block), the
// minimums off with one more MFMA a super-block.  Rows past the last are read as the last (the same lines again) and never stored.
#include "blocks.hpp"
#include "few_rule.hpp"
#include "gemm_few.hpp"

#include <cmath>
#include <cstdlib>

namespace nh {

namespace {

typedef const __attribute__((address_space(1))) u32x4 *global_uint4;
typedef uint32_t u32x4_loose __attribute__((ext_vector_type(4), aligned(4)));
typedef const __attribute__((address_space(1))) u32x4_loose *global_loose4;
typedef uint32_t u32_half __attribute__((aligned(2)));
typedef const __attribute__((address_space(1))) u32_half *global_word_at_half;
typedef const __attribute__((address_space(1))) uint16_t *global_half_word;

__device__ __forceinline__ half2_t as_halves(uint32_t v) { return __builtin_bit_cast(half2_t, v); }
__device__ __forceinline__ uint32_t as_word(half2_t v) { return __builtin_bit_cast(uint32_t, v); }

// low lanes (part 0) get the other part's `a`, high lanes (part 1) the other part's `b`
__device__ __forceinline__ uint32_t crossed(uint32_t a, uint32_t b, uint32_t part) {
    const auto swapped = __builtin_amdgcn_permlane32_swap(a, b, false, false);  // exchanges a's high lanes with b's low lanes
    return part ? swapped[0] : swapped[1];
}

// the 16 bytes of a run that starts `shift` bits (0 or 16) into `low`; `above` holds the half word behind `low` in its low bits
__device__ __forceinline__ u32x4 placed(const u32x4 &low, uint32_t above, uint32_t shift) {
    return u32x4{__builtin_amdgcn_alignbit(low.y, low.x, shift), __builtin_amdgcn_alignbit(low.z, low.y, shift),
                 __builtin_amdgcn_alignbit(low.w, low.z, shift), __builtin_amdgcn_alignbit(above, low.w, shift)};
}

// four stored bytes (each below 1024 as a half) as halves less `bias`, in the order 0, 2 then 1, 3
__device__ __forceinline__ void bytes_as_halves(uint32_t bytes, half2_t bias, half2_t &even, half2_t &odd) {
    even = as_halves(__builtin_amdgcn_perm(0u, bytes, 0x0c020c00u) | 0x64006400u) - bias;
    odd = as_halves(__builtin_amdgcn_perm(0u, bytes, 0x0c030c01u) | 0x64006400u) - bias;
}

// ---- what a lane holds of one column's super-block, and the B operands it makes of it -----------------------------------
// fetch(): the loads.  ready(): once a super-block.  operand(g, depth): numbers 64 g + 32 (depth / 2) + 16 part + 8 (depth % 2) ...
// PLANES operands add up to the weight (over d).

template <bool FIFTH>
struct FewQ45 {
    static constexpr int STEPS = 4, PLANES = 1, CLOSED = 4;
    static constexpr uint32_t BYTES = FIFTH ? 176u : 144u;
    static constexpr bool FLOORS = true;
    static constexpr float CENTRE = FIFTH ? 16.0f : 8.0f;
    u32x4 header, fifth, runs[4];
    half2_t low_scale, high_scale, low_centre, high_centre;
    __device__ __forceinline__ void fetch(const uint8_t *row, uint32_t unit, uint32_t, uint32_t part) {
        const uint8_t *block = row + (size_t)unit * BYTES;
        header = *(global_uint4)(uintptr_t)block;
        if (FIFTH) fifth = *(global_uint4)(uintptr_t)(block + 16u + 16u * part);
#pragma unroll
        for (int g = 0; g < 4; g++) runs[g] = *(global_uint4)(uintptr_t)(block + (FIFTH ? 48u : 16u) + 32u * g + 16u * part);
    }
    // A sub-block whose minimum is zero is left as it lies: its weights may be exact zeros, and beside a large activation that
    // meets one, the centre's share and what takes it off again would swallow the other numbers' products (0x3f + 0x7f stays below 0x100:
    // no carry crosses a byte)
    __device__ __forceinline__ uint32_t centred(int high) const {  // 0xff where a sub-block's codes are centred, of four sub-blocks
        const uint32_t minimums = high ? ((header.w >> 4) & 0x0f0f0f0fu) | ((header.z >> 2) & 0x30303030u) : header.z & 0x3f3f3f3fu;
        const uint32_t some = (minimums + 0x7f7f7f7fu) & 0x80808080u;
        return some | (some - (some >> 7));
    }
    __device__ __forceinline__ float scale() const { return (float)as_halves(header.x).x * 16384.0f; }  // operands are code * sc * 2^-14
    __device__ __forceinline__ float floor_scale() const { return (float)as_halves(header.x).y * -64.0f; }  // the sums are packed / 64
    __device__ __forceinline__ float centre_scale() const { return (float)as_halves(header.x).x * (64.0f * CENTRE); }
    // the eight minimums (`scales`: the eight scales where the codes are centred) as halves; k 8..15 meet the sums' residues * 2^11
    __device__ __forceinline__ half8_t floors(uint32_t part, bool scales) const {
        const half2_t offset = {(_Float16)1024.0f, (_Float16)1024.0f};
        const uint32_t first = scales ? header.y : header.z, more = scales ? header.w : header.w >> 4;
        const uint32_t lo4 = first & 0x3f3f3f3fu & (scales ? centred(0) : ~0u), hi4 = ((more & 0x0f0f0f0fu) | ((first >> 2) & 0x30303030u)) & (scales ? centred(1) : ~0u);
        half2_t m[4] = {as_halves(__builtin_amdgcn_perm(0u, lo4, 0x0c010c00u) | 0x64006400u) - offset,
                        as_halves(__builtin_amdgcn_perm(0u, lo4, 0x0c030c02u) | 0x64006400u) - offset,
                        as_halves(__builtin_amdgcn_perm(0u, hi4, 0x0c010c00u) | 0x64006400u) - offset,
                        as_halves(__builtin_amdgcn_perm(0u, hi4, 0x0c030c02u) | 0x64006400u) - offset};
        const _Float16 down = part ? (_Float16)0.00048828125f : (_Float16)1.0f;
        const half2_t downs = {down, down};
        return __builtin_bit_cast(half8_t, u32x4{as_word(m[0] * downs), as_word(m[1] * downs), as_word(m[2] * downs), as_word(m[3] * downs)});
    }
    __device__ __forceinline__ void step(int g) {
        // 6-bit scales of sub-blocks 2g, 2g + 1 (crates/neura-precision/src/ggml.rs:127-136); 0x6400 | v is the half 1024 + v
        const half2_t offset = {(_Float16)1024.0f, (_Float16)1024.0f}, powers = {(_Float16)1024.0f, (_Float16)64.0f};
        const uint32_t shift = 16u * (g & 1);
        const uint32_t ya = (header.y >> shift) & 0xffffu, wa = (header.w >> shift) & 0xffffu;
        const uint32_t sc = g < 2 ? (ya & 0x3f3fu) : ((wa & 0x0f0fu) | ((ya >> 2) & 0x3030u));
        const half2_t scales = (as_halves(__builtin_amdgcn_perm(0u, sc, 0x0c010c00u) | 0x64006400u) - offset) * powers;  // (sc0 * 2^10, sc1 * 2^6)
        low_scale = half2_t{scales.x, scales.x}, high_scale = half2_t{scales.y, scales.y};
        // a code enters less CENTRE: the products then add up to sums of the output's own size, and not to ones that the minimums
        // take most of off again (2-norm from the exact products, eight rows of the 7B shapes: 2.2e-7 -> 1.1e-7); CENTRE times
        // the scales comes back with the minimums.  (code - CENTRE) * sc * 2^-14 is exact: one rounding, of a whole number below 2^11
        const half2_t down = {(_Float16)(-CENTRE * 0.00006103515625f), (_Float16)(-CENTRE * 0.00006103515625f)};
        const uint32_t some = sc & (centred(g >> 1) >> shift);
        const half2_t centres = (as_halves(__builtin_amdgcn_perm(0u, some, 0x0c010c00u) | 0x64006400u) - offset) * down;
        low_centre = half2_t{centres.x, centres.x}, high_centre = half2_t{centres.y, centres.y};
    }
    __device__ __forceinline__ void operand(int g, int depth, half8_t (&b)[PLANES]) const {
        const uint32_t words[4] = {runs[g].x, runs[g].y, runs[g].z, runs[g].w}, fifths[4] = {fifth.x, fifth.y, fifth.z, fifth.w};
        uint32_t out[4];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const int at = 2 * (depth & 1) + w;
            const uint32_t mask = depth < 2 ? 0x000f000fu : 0x00f000f0u;
            uint32_t even = words[at] & mask, odd = (words[at] >> 8) & mask;
            if (FIFTH) {
                // bit 2g of a byte to bit 4 of its lane (beside the low nibble), bit 2g + 1 to bit 8 (beside the high nibble's four)
                const uint32_t bits = fifths[at] >> (2 * g + (depth < 2 ? 0 : 1));
                even |= (bits & 0x00010001u) << (depth < 2 ? 4 : 8), odd |= ((bits >> 8) & 0x00010001u) << (depth < 2 ? 4 : 8);
            }
            const half2_t scale = depth < 2 ? low_scale : high_scale, centre = depth < 2 ? low_centre : high_centre;
            out[2 * w] = as_word(__builtin_elementwise_fma(as_halves(even), scale, centre)), out[2 * w + 1] = as_word(__builtin_elementwise_fma(as_halves(odd), scale, centre));
        }
        b[0] = __builtin_bit_cast(half8_t, u32x4{out[0], out[1], out[2], out[3]});
    }
};

// 210-byte blocks on any half word: thirteen 16-byte pieces in a row (eight of nibbles, four of bit pairs, the scales), of which
// part p takes every second one.  Each is read from the 4-byte boundary below it; the half word it then lacks is the first one the
// next piece's load holds, in the other part's lanes.
struct FewQ6 {
    static constexpr int CLOSED = 2;              // (sums of sc * q reach further than the others': weighed by d twice a super-block)
    static constexpr int STEPS = 4, PLANES = 2;  // sc = 16 (sc >> 4) + (sc & 15): both products with a code are exact halves
    static constexpr uint32_t BYTES = 210u;
    static constexpr bool FLOORS = false;
    u32x4 pieces[7];  // nibbles 0..3, bit pairs 4, 5; the scales
    uint32_t tail;    // bytes 206..209: the half word above the scales, d
    uint32_t scales[4];
    __device__ __forceinline__ void fetch(const uint8_t *row, uint32_t unit, uint32_t, uint32_t part) {
        const uint8_t *block = row + (size_t)unit * BYTES;
#pragma unroll
        for (int i = 0; i < 6; i++) pieces[i] = *(global_loose4)((uintptr_t)(block + 32u * i + 16u * part) & ~(uintptr_t)3);
        pieces[6] = *(global_loose4)((uintptr_t)(block + 192u) & ~(uintptr_t)3);
        tail = *(global_word_at_half)(uintptr_t)(block + 206u);
    }
    __device__ __forceinline__ void ready(const uint8_t *row, uint32_t unit, uint32_t part) {
        const uint32_t shift = (uint32_t)((uintptr_t)(row + (size_t)unit * BYTES) & 2u) * 8u;
        const u32x4 sc = placed(pieces[6], tail, shift);
        // a lane's scales are those of its 16-number groups: bytes part, part + 2 of every word come down to bytes 0 and 2
        scales[0] = sc.x >> (8u * part), scales[1] = sc.y >> (8u * part), scales[2] = sc.z >> (8u * part), scales[3] = sc.w >> (8u * part);
        uint32_t above[6];
#pragma unroll
        for (int i = 0; i < 5; i++) above[i] = crossed(pieces[i].x, pieces[i + 1].x, part);
        const uint32_t last = crossed(pieces[5].x, pieces[5].x, part);
        above[5] = part ? pieces[6].x : last;
#pragma unroll
        for (int i = 0; i < 6; i++) pieces[i] = placed(pieces[i], above[i], shift);
    }
    __device__ __forceinline__ float scale() const { return (float)as_halves(tail).y; }
    __device__ __forceinline__ void step(int) {}
    __device__ __forceinline__ void operand(int g, int depth, half8_t (&b)[PLANES]) const {
        const int n = g >> 1, quarter = 2 * (g & 1) + (depth >> 1);  // numbers 128 n + 32 quarter + ..
        const half2_t bias = {(_Float16)1056.0f, (_Float16)1056.0f};  // a code is stored 32 too large
        const int sc = __builtin_amdgcn_sbfe((int)scales[g], 16u * (depth >> 1), 8u);
        const _Float16 fine = (_Float16)(float)(sc & 15), coarse = (_Float16)(float)(16 * (sc >> 4));
        const half2_t fine2 = {fine, fine}, coarse2 = {coarse, coarse};
        const u32x4 nibbles = pieces[2 * n + (quarter & 1)], pairs = pieces[4 + n];
        const uint32_t nibble_words[4] = {nibbles.x, nibbles.y, nibbles.z, nibbles.w}, pair_words[4] = {pairs.x, pairs.y, pairs.z, pairs.w};
        uint32_t one[4], two[4];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const int at = 2 * (depth & 1) + w;
            const uint32_t low4 = (quarter >= 2 ? nibble_words[at] >> 4 : nibble_words[at]) & 0x0f0f0f0fu;
            half2_t even, odd;
            bytes_as_halves(low4 | (((pair_words[at] >> (2 * quarter)) & 0x03030303u) << 4), bias, even, odd);
            one[2 * w] = as_word(even * fine2), one[2 * w + 1] = as_word(odd * fine2);
            two[2 * w] = as_word(even * coarse2), two[2 * w + 1] = as_word(odd * coarse2);
        }
        b[0] = __builtin_bit_cast(half8_t, u32x4{one[0], one[1], one[2], one[3]});
        b[1] = __builtin_bit_cast(half8_t, u32x4{two[0], two[1], two[2], two[3]});
    }
};

// 110-byte blocks on any half word: two 16-byte pieces of third bits, four of bit pairs, then twelve bytes of scales and d; read as
// Q6_K's.  (sc - 32) * (code - 4) stays within +-128: one exact plane.
struct FewQ3 {
    static constexpr int STEPS = 4, PLANES = 1, CLOSED = 4;
    static constexpr uint32_t BYTES = 110u;
    static constexpr bool FLOORS = false;
    u32x4 pieces[3], tail;  // third bits, bit pairs of both halves; 16 bytes from the 4-byte boundary below byte 94
    uint32_t d;
    uint32_t nibbles[2], tops;
    half2_t first_scale, second_scale;
    __device__ __forceinline__ void fetch(const uint8_t *row, uint32_t unit, uint32_t, uint32_t part) {
        const uint8_t *block = row + (size_t)unit * BYTES;
#pragma unroll
        for (int i = 0; i < 3; i++) pieces[i] = *(global_loose4)((uintptr_t)(block + 32u * i + 16u * part) & ~(uintptr_t)3);
        tail = *(global_loose4)((uintptr_t)(block + 94u) & ~(uintptr_t)3);
        d = *(global_half_word)(uintptr_t)(block + 108u);
    }
    __device__ __forceinline__ void ready(const uint8_t *row, uint32_t unit, uint32_t part) {
        const uint32_t shift = (uint32_t)((uintptr_t)(row + (size_t)unit * BYTES) & 2u) * 8u;
        uint32_t above[3];
#pragma unroll
        for (int i = 0; i < 2; i++) above[i] = crossed(pieces[i].x, pieces[i + 1].x, part);
        const uint32_t last = crossed(pieces[2].x, pieces[2].x, part);
        above[2] = part ? tail.x : last;  // (wanted on an odd half word: the tail then starts at byte 94)
#pragma unroll
        for (int i = 0; i < 3; i++) pieces[i] = placed(pieces[i], above[i], shift);
        // bytes 96..107; a lane's scales are those of its 16-number groups
        const uint32_t words[3] = {shift ? __builtin_amdgcn_alignbit(tail.y, tail.x, 16u) : tail.y, shift ? __builtin_amdgcn_alignbit(tail.z, tail.y, 16u) : tail.z,
                                   shift ? __builtin_amdgcn_alignbit(tail.w, tail.z, 16u) : tail.w};
        nibbles[0] = words[0] >> (8u * part), nibbles[1] = words[1] >> (8u * part), tops = words[2] >> (8u * part);
    }
    __device__ __forceinline__ float scale() const { return (float)__builtin_bit_cast(_Float16, (uint16_t)d); }
    __device__ __forceinline__ void step(int g) {
        // scales 4 g + part and 4 g + 2 + part: nibbles of bytes 0 and 2 (the low ones for the first eight), top bits at 2 g
        const half2_t bias = {(_Float16)1056.0f, (_Float16)1056.0f};  // 0x6400 | v is the half 1024 + v; a scale is stored 32 too large
        const uint32_t two = nibbles[g & 1];
        const uint32_t pair = ((g < 2 ? two : two >> 4) & 0x000f000fu) | (((tops >> (2 * g)) & 0x00030003u) << 4);
        const half2_t scales = as_halves(pair | 0x64006400u) - bias;
        first_scale = half2_t{scales.x, scales.x}, second_scale = half2_t{scales.y, scales.y};
    }
    __device__ __forceinline__ void operand(int g, int depth, half8_t (&b)[PLANES]) const {
        const int n = g >> 1, j = 2 * (g & 1) + (depth >> 1);
        const half2_t bias = {(_Float16)1028.0f, (_Float16)1028.0f};  // a code is stored 4 too large
        const u32x4 third = pieces[0], pairs = pieces[1 + n];
        const uint32_t third_words[4] = {third.x, third.y, third.z, third.w}, pair_words[4] = {pairs.x, pairs.y, pairs.z, pairs.w};
        const half2_t scale = depth < 2 ? first_scale : second_scale;
        uint32_t out[4];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const int at = 2 * (depth & 1) + w;
            half2_t even, odd;
            bytes_as_halves(((pair_words[at] >> (2 * j)) & 0x03030303u) | (((third_words[at] >> (4 * n + j)) & 0x01010101u) << 2), bias, even, odd);
            out[2 * w] = as_word(even * scale), out[2 * w + 1] = as_word(odd * scale);
        }
        b[0] = __builtin_bit_cast(half8_t, u32x4{out[0], out[1], out[2], out[3]});
    }
};

// 34-byte blocks on any half word, two steps (four blocks) at a time; K is a multiple of 64, so the last unit may be one step: its
// second is read as the first and weighed by zero.  Part 0 holds a block's d in its half word, part 1 the half word behind the block's
// codes; each needs the other's.  The scale cannot ride in the operand: the sums are weighed a block.
struct FewQ8 {
    static constexpr int STEPS = 2, PLANES = 1, CLOSED = 2;
    static constexpr uint32_t BYTES = 68u;  // of a step
    static constexpr bool FLOORS = false;
    u32x4 codes[4];
    uint32_t ends[4];
    __device__ __forceinline__ void fetch(const uint8_t *row, uint32_t unit, uint32_t steps, uint32_t part) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint8_t *block = row + (size_t)min(2u * unit + (i >> 1), steps - 1u) * BYTES + 34u * (i & 1);
            codes[i] = *(global_loose4)((uintptr_t)(block + 2u + 16u * part) & ~(uintptr_t)3);
            ends[i] = *(global_half_word)(uintptr_t)(block + 32u * part);
        }
    }
    __device__ __forceinline__ void ready(const uint8_t *row, uint32_t unit, uint32_t steps, uint32_t part) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t step = 2u * unit + (i >> 1);
            // the codes of part 0 start two bytes behind the block, on a word boundary where the block is not
            const uint32_t shift = 16u - (uint32_t)((uintptr_t)(row + (size_t)min(step, steps - 1u) * BYTES + 34u * (i & 1)) & 2u) * 8u;
            const uint32_t other = crossed(codes[i].x, ends[i], part);  // part 0: part 1's first word; part 1: part 0's d
            codes[i] = placed(codes[i], part ? ends[i] : other, shift);
            ends[i] = step < steps ? (part ? other : ends[i]) : 0u;
        }
    }
    __device__ __forceinline__ float block_scale(int i) const { return (float)__builtin_bit_cast(_Float16, (uint16_t)ends[i]); }
    __device__ __forceinline__ void step(int) {}
    __device__ __forceinline__ void operand(int g, int depth, half8_t (&b)[PLANES]) const {
        const half2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};  // a signed byte with its top bit flipped is 128 too large
        const u32x4 run = codes[2 * g + (depth >> 1)];
        const uint32_t words[4] = {run.x, run.y, run.z, run.w};
        uint32_t out[4];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            half2_t even, odd;
            bytes_as_halves(words[2 * (depth & 1) + w] ^ 0x80808080u, bias, even, odd);
            out[2 * w] = as_word(even), out[2 * w + 1] = as_word(odd);
        }
        b[0] = __builtin_bit_cast(half8_t, u32x4{out[0], out[1], out[2], out[3]});
    }
};

template <int ELEMENT>
struct FewOf;
template <> struct FewOf<NH_Q4_K> { typedef FewQ45<false> type; };
template <> struct FewOf<NH_Q5_K> { typedef FewQ45<true> type; };
template <> struct FewOf<NH_Q6_K> { typedef FewQ6 type; };
template <> struct FewOf<NH_Q3_K> { typedef FewQ3 type; };
template <> struct FewOf<NH_Q8_0> { typedef FewQ8 type; };

constexpr uint32_t FEW_SLICES_MOST = 8;

// what an activation row's numbers beyond its packed pieces add to an output -- or, where they are too many, take its place: numbers
// and weights as they are stored, added in 64 bits
template <int ELEMENT>
__device__ __forceinline__ float beyond_pieces(float value, const WholeRow &held, const float *outside, const uint8_t *row, uint32_t K) {
    bool all = false;
    for (uint32_t part = 0; part < WHOLE_PARTS; part++) all |= held.listed[part] > WHOLE_LISTED;
    double sum = all ? 0.0 : (double)value;
    if (all) {
        for (uint32_t k = 0; k < K; k++) sum = fma((double)outside[k], (double)stored_element<ELEMENT>(row, k), sum);
    } else {
        for (uint32_t part = 0; part < WHOLE_PARTS; part++)
            for (uint32_t i = 0; i < held.listed[part]; i++) sum = fma((double)held.list[part][i].value, (double)stored_element<ELEMENT>(row, held.list[part][i].k), sum);
    }
    return (float)sum;
}

// where piece j of a tile's activation row r lies among the sums of a 32 x 32 block, [q][part][column][4]: q and the rest at column 0
struct PieceRow {
    uint32_t q, seat;
};
__device__ __forceinline__ PieceRow piece_row(uint32_t r, uint32_t j) {
    const uint32_t row = WHOLE_PIECES * r + j;
    return {row >> 3, ((row >> 2) & 1u) * 128u + (row & 3u)};
}

// MT: tiles of 32 packed rows a wave multiplies its weights by; GATED: a wave walks the same 32 columns of the gate and of the up
// matrix, and what leaves is silu(gate) * up; AHEAD: steps the activation operands are read ahead (the loads of a wave come
// back in order: an operand asked for after the next super-block's weights waits for them, so they are asked for
// early enough to be waited on late).
template <int ELEMENT, int MT, bool GATED, int AHEAD>
__global__ __launch_bounds__(512) void gemm_few_kernel(FewParams p) {
    typedef typename FewOf<ELEMENT>::type Weights;
    constexpr int NT = GATED ? 2 : 1, STEPS = Weights::STEPS;
    static_assert(AHEAD % STEPS == 0 || STEPS % AHEAD == 0, "a step's slot is its number within a unit");
    constexpr int SLOTS = AHEAD < STEPS ? AHEAD : STEPS;
    static_assert(SLOTS == AHEAD, "operands are read at most one unit ahead");
    extern __shared__ __attribute__((aligned(16))) uint8_t few_lds[];
    float4 *parts = reinterpret_cast<float4 *>(few_lds);  // [wave][NT][MT][4][64]
    const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, part = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t shares = p.deep * p.slices, share = blockIdx.z * p.deep + wave;
    const uint32_t n0 = blockIdx.x * FEW_TILE, tile0 = blockIdx.y * MT;
    const uint32_t steps = p.K / 64u, units = (steps + STEPS - 1u) / STEPS;
    const uint32_t nsb = p.K / 256u;

    const uint32_t column = min(n0 + l32, p.N - 1u);
    const uint8_t *wrow[NT];
    if (GATED) {
        wrow[0] = p.W + (size_t)column * p.row_bytes, wrow[NT - 1] = p.W1 + (size_t)column * p.row_bytes;
    } else {
        // a tile lies in one matrix: the boundaries between stacked matrices are multiples of the tile
        wrow[0] = column < p.end0   ? p.W + (size_t)column * p.row_bytes
                  : column < p.end1 ? p.W1 + (size_t)(column - p.end0) * p.row_bytes
                                    : p.W2 + (size_t)(column - p.end1) * p.row_bytes;
    }
    const _Float16 *arow[MT], *srow[MT];
    const uint32_t last_tile = (p.rows - 1u) >> 5;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const uint32_t tile = min(tile0 + i, last_tile);
        const uint32_t at = (part * 32u + min(l32, p.rows - 1u - 32u * tile)) * 8u;
        arow[i] = p.A + (size_t)tile * steps * 2048u + at;
        srow[i] = p.S + (size_t)tile * nsb * 512u + at;
    }

    f32x16 acc[NT][MT], zero;
#pragma unroll
    for (int e = 0; e < 16; e++) zero[e] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[t][i] = zero;

    half8_t a[SLOTS][4][MT];
    auto fetch_rows = [&](int slot, int depth, uint32_t step) {
        const size_t at = (size_t)min(step, steps - 1u) * 2048u + 512u * depth;
#pragma unroll
        for (int i = 0; i < MT; i++) a[slot][depth][i] = __builtin_bit_cast(half8_t, *(global_uint4)(uintptr_t)(arow[i] + at));
    };
    // a whole row's scale and whether it lists numbers: asked for before the weights and put by for the end
    __shared__ float2 heads[MT * WHOLE_TILE];
    if (p.pieces == WHOLE_PIECES && threadIdx.x < MT * WHOLE_TILE) {
        const u32x4 head = *(global_uint4)(uintptr_t)(p.whole + min(tile0 * WHOLE_TILE + threadIdx.x, p.M - 1u));
        heads[threadIdx.x] = float2{__builtin_bit_cast(float, head.x), __builtin_bit_cast(float, head.z | head.w)};
    }
    if (share < units) {
        Weights next[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) next[t].fetch(wrow[t], share, steps, part);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < SLOTS; s++)
#pragma unroll
            for (int depth = 0; depth < 4; depth++) fetch_rows(s, depth, share * STEPS + s);
        for (uint32_t unit = share; unit < units; unit += shares) {
            Weights w[NT];
            half8_t sums[MT];
            const uint32_t after = min(unit + shares, units - 1u);  // past the end the last unit again, dropped
#pragma unroll
            for (int t = 0; t < NT; t++) w[t] = next[t];
            if (Weights::FLOORS) {
#pragma unroll
                for (int i = 0; i < MT; i++) sums[i] = __builtin_bit_cast(half8_t, *(global_uint4)(uintptr_t)(srow[i] + (size_t)unit * 512u));
            }
#pragma unroll
            for (int t = 0; t < NT; t++) next[t].fetch(wrow[t], after, steps, part);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if constexpr (ELEMENT == NH_Q8_0) w[t].ready(wrow[t], unit, steps, part);
                else if constexpr (ELEMENT == NH_Q6_K || ELEMENT == NH_Q3_K) w[t].ready(wrow[t], unit, part);
            }
            f32x16 tmp[NT][MT];
#pragma unroll
            for (int g = 0; g < STEPS; g++) {
                const int slot = g % SLOTS;
#pragma unroll
                for (int t = 0; t < NT; t++) w[t].step(g);
#pragma unroll
                for (int depth = 0; depth < 4; depth++) {
                    const bool first = ELEMENT == NH_Q8_0 ? (depth & 1) == 0 : (g % Weights::CLOSED == 0 && depth == 0);
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        half8_t b[Weights::PLANES];
                        w[t].operand(g, depth, b);
#pragma unroll
                        for (int i = 0; i < MT; i++) {
                            tmp[t][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[slot][depth][i], b[0], first ? zero : tmp[t][i], 0, 0, 0);
                            if (Weights::PLANES > 1)
                                tmp[t][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[slot][depth][i], b[Weights::PLANES - 1], tmp[t][i], 0, 0, 0);
                        }
                    }
                    // these registers are free: the same operands of the step AHEAD of this one
                    fetch_rows(slot, depth, (g + AHEAD < STEPS ? unit : after) * STEPS + (g + AHEAD) % STEPS);
                    if constexpr (ELEMENT == NH_Q8_0) {
                        if (depth & 1) {
#pragma unroll
                            for (int t = 0; t < NT; t++) {
                                const float scale = w[t].block_scale(2 * g + (depth >> 1));
#pragma unroll
                                for (int i = 0; i < MT; i++)
#pragma unroll
                                    for (int e = 0; e < 16; e++) acc[t][i][e] = fmaf(scale, tmp[t][i][e], acc[t][i][e]);
                            }
                        }
                    }
                }
                if constexpr (ELEMENT != NH_Q8_0) {
                    if ((g + 1) % Weights::CLOSED == 0) {
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            const float scale = w[t].scale();
#pragma unroll
                            for (int i = 0; i < MT; i++)
#pragma unroll
                                for (int e = 0; e < 16; e++) acc[t][i][e] = fmaf(scale, tmp[t][i][e], acc[t][i][e]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (Weights::FLOORS) {
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const half8_t b = w[t].floors(part, false), c = w[t].floors(part, true);
                    const float floor_scale = w[t].floor_scale(), centre_scale = w[t].centre_scale();
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const f32x16 floors = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[i], b, zero, 0, 0, 0);
                        const f32x16 centres = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[i], c, zero, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 16; e++) acc[t][i][e] += fmaf(floor_scale, floors[e], centre_scale * centres[e]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                parts[(((wave * NT + t) * MT + i) * 4u + q) * 64u + lane] = float4{acc[t][i][4 * q], acc[t][i][4 * q + 1], acc[t][i][4 * q + 2], acc[t][i][4 * q + 3]};
    __syncthreads();
    // ---- out: an item is column l32 and rows 8q + 4 part .. + 3 of a 32 x 32 block; the shares of K are added in their order
    constexpr uint32_t items = MT * 256u;
    auto own_sum = [&](uint32_t item, int t) {
        const uint32_t at = item & 63u, q = (item >> 6) & 3u, i = item >> 8;
        float4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t s = 0; s < p.deep; s++) {
            const float4 add = parts[(((s * NT + t) * MT + i) * 4u + q) * 64u + at];
            v.x += add.x, v.y += add.y, v.z += add.z, v.w += add.w;
        }
        return v;
    };
    auto row_of = [&](uint32_t item) { return (tile0 + (item >> 8)) * FEW_TILE + 8u * ((item >> 6) & 3u) + 4u * ((item >> 5) & 1u); };
    // with more workgroups over the same outputs: each leaves its sums in memory and the last to arrive adds them, in the order of
    // the slices, so the sums do not depend on who that is.  Nobody waits for another.
    typedef unsigned long long pair_word;
    auto place_of = [&](uint32_t slice, uint32_t item, int t) {
        const size_t place = ((size_t)slice * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
        return reinterpret_cast<pair_word *>(p.partial) + ((place * items + item) * NT + t) * 2u;
    };
    if (p.slices > 1u) {
        for (uint32_t item = threadIdx.x; item < items; item += blockDim.x) {
            if (row_of(item) >= p.rows) continue;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const float4 v = own_sum(item, t);
                pair_word *to = place_of(blockIdx.z, item, t);
                __hip_atomic_store(to, __builtin_bit_cast(pair_word, float2{v.x, v.y}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(to + 1, __builtin_bit_cast(pair_word, float2{v.z, v.w}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        // the stores go past the caches that other workgroups do not share, and the loads below come from there: what is left to
        // order is their completion (a fence would write back and drop whole caches: 20 to 90 us a launch)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // (every wave's sums are out, and the last word of LDS read)
        uint32_t *arrived = reinterpret_cast<uint32_t *>(few_lds), *meet = p.meets + blockIdx.y * gridDim.x + blockIdx.x;
        if (threadIdx.x == 0) arrived[0] = __hip_atomic_fetch_add(meet, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (arrived[0] != p.slices - 1u) return;
        asm volatile("" ::: "memory");
        if (threadIdx.x == 0) __hip_atomic_store(meet, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // as the next launch expects it
    }
    auto leave = [&](uint32_t m, uint32_t n, float value, float up) {
        if (m >= p.M) return;
        if (GATED) value = value * (1.0f / (1.0f + expf(-value))) * up;
        const size_t to = (size_t)m * p.ldy + n;
        p.Y[to] = p.residual ? p.residual[to] + value : value;
    };
    if (p.pieces == WHOLE_PIECES) {
        // an item is a column and one of a tile's ten activation rows, whose pieces lie wherever rows 3r .. 3r + 2 do
        const uint32_t rows = min(p.M, WHOLE_TILE), outputs = MT * rows * 32u;
        for (uint32_t item = threadIdx.x; item < outputs; item += blockDim.x) {
            const uint32_t at = item & 31u, i = (item >> 5) / rows, r = (item >> 5) - i * rows;
            const uint32_t m = (tile0 + i) * WHOLE_TILE + r, n = n0 + at;
            if (n >= p.N || m >= p.M) continue;
            const float2 head = heads[i * WHOLE_TILE + r];
            float out[NT], v[NT][WHOLE_PIECES];
            // (every load of a share's sums before any is added: a chain of them is an LDS latency each)
            if (p.slices == 1u) {
                const float *sums = reinterpret_cast<const float *>(few_lds);
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (uint32_t j = 0; j < WHOLE_PIECES; j++) v[t][j] = 0.0f;
                for (uint32_t s = 0; s < p.deep; s++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
#pragma unroll
                        for (uint32_t j = 0; j < WHOLE_PIECES; j++) v[t][j] += sums[(((s * NT + t) * MT + i) * 4u + piece_row(r, j).q) * 256u + piece_row(r, j).seat + at * 4u];
            } else {
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (uint32_t j = 0; j < WHOLE_PIECES; j++) {
                        uint32_t held[FEW_SLICES_MOST];
#pragma unroll
                        for (uint32_t s = 0; s < FEW_SLICES_MOST; s++)
                            held[s] = __hip_atomic_load(reinterpret_cast<const uint32_t *>(place_of(min(s, p.slices - 1u), i * 256u + piece_row(r, j).q * 64u + piece_row(r, j).seat / 4u + at, t)) +
                                                            piece_row(r, j).seat % 4u,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        v[t][j] = 0.0f;
#pragma unroll
                        for (uint32_t s = 0; s < FEW_SLICES_MOST; s++)
                            if (s < p.slices) v[t][j] += __builtin_bit_cast(float, held[s]);
                    }
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                out[t] = fmaf(fmaf(v[t][2], 0.00048828125f, v[t][1]), 0.00048828125f, v[t][0]) * head.x;
                if (__builtin_bit_cast(uint32_t, head.y)) {
                    const uint8_t *from = GATED        ? (t ? p.W1 : p.W) + (size_t)n * p.row_bytes
                                          : n < p.end0 ? p.W + (size_t)n * p.row_bytes
                                          : n < p.end1 ? p.W1 + (size_t)(n - p.end0) * p.row_bytes
                                                       : p.W2 + (size_t)(n - p.end1) * p.row_bytes;
                    out[t] = beyond_pieces<ELEMENT>(out[t], p.whole[m], p.outside + (size_t)m * p.K, from, p.K);
                }
            }
            leave(m, n, out[0], out[NT - 1]);
        }
        return;
    }
    for (uint32_t item = threadIdx.x; item < items; item += blockDim.x) {
        const uint32_t row = row_of(item), n = n0 + (item & 31u);
        if (n >= p.N || row >= p.rows) continue;
        float v[NT][4];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            v[t][0] = v[t][1] = v[t][2] = v[t][3] = 0.0f;
            if (p.slices == 1u) {
                const float4 sum = own_sum(item, t);
                v[t][0] = sum.x, v[t][1] = sum.y, v[t][2] = sum.z, v[t][3] = sum.w;
            } else {
                pair_word held[FEW_SLICES_MOST][2];
#pragma unroll
                for (uint32_t s = 0; s < FEW_SLICES_MOST; s++) {
                    const pair_word *from = place_of(min(s, p.slices - 1u), item, t);
                    held[s][0] = __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    held[s][1] = __hip_atomic_load(from + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for (uint32_t s = 0; s < FEW_SLICES_MOST; s++) {
                    if (s >= p.slices) break;
                    const float2 low = __builtin_bit_cast(float2, held[s][0]), high = __builtin_bit_cast(float2, held[s][1]);
                    v[t][0] += low.x, v[t][1] += low.y, v[t][2] += high.x, v[t][3] += high.y;
                }
            }
        }
        if (p.pieces == 2u) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const uint32_t m = (row >> 1) + e;
                const float unscale = p.unscale[min(m, p.M - 1u)];
                leave(m, n, fmaf(v[0][2 * e + 1], 0.00048828125f, v[0][2 * e]) * unscale, fmaf(v[NT - 1][2 * e + 1], 0.00048828125f, v[NT - 1][2 * e]) * unscale);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) leave(row + e, n, v[0][e], v[NT - 1][e]);
        }
    }
}

constexpr uint32_t slice_list[] = {1, 2, 3, 4, 6, 8};

template <int ELEMENT, int MT, bool GATED>
int32_t launch_few(nh_device *d, FewParams p) {
    constexpr int STEPS = FewOf<ELEMENT>::type::STEPS;
    constexpr int NT = GATED ? 2 : 1;
    constexpr int AHEAD = MT * NT > 2 ? 1 : (STEPS < 4 || MT * NT > 1 ? 2 : 4);
    const uint32_t units = (p.K / 64u + STEPS - 1u) / STEPS, tiles = (p.N + FEW_TILE - 1u) / FEW_TILE, row_tiles = (p.rows + FEW_TILE - 1u) / FEW_TILE;
    // the split of a workgroup's waves that walks the fewest units: rounds of workgroups times the units of a wave (and what a
    // workgroup takes before its first and after its last, about two units' time).  A matrix of few tiles and deep rows leaves most
    // of the chip idle that way, so K may be shared among workgroups too: their meeting costs a unit's time and the passage of
    // their sums, 2.5 MB in another (eight rows of fp32, with the packing: ffn_down of the 7B shape Q8_0 55 -> 37 us, Q6_K
    // 45 -> 34, Q5_K 37 -> 29, of the 1.5B shape Q8_0 28 -> 18; gate|up of the 7B shape, 592 tiles, is better left alone: Q4_K 34, not 38)
    uint32_t best = ~0u;
    const uint32_t places = tiles * ((row_tiles + MT - 1u) / MT);
    for (uint32_t deep = 1; deep <= 8u; deep++)
        for (uint32_t slices : slice_list) {
            const uint32_t resident = (uint32_t)d->compute_units * (8u / deep);
            if (slices > 1u && (places > FEW_MEETS || deep * slices > units || (size_t)slices * places * MT * NT * 4096u > FEW_PARTIAL_BYTES)) continue;
            const uint32_t meeting = slices > 1u ? 64u + (uint32_t)((uint64_t)slices * p.N * NT * p.rows * 4u * 64u / 2500000u) : 0u;
            const uint32_t cost = ((places * slices + resident - 1u) / resident) * ((units + deep * slices - 1u) / (deep * slices) + 2u) * 64u + meeting + deep;
            if (cost < best) best = cost, p.deep = deep, p.slices = slices;
        }
    const size_t lds = (size_t)p.deep * NT * MT * 4096u;
    static bool sized = false;
    if (!sized) {
        NH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_few_kernel<ELEMENT, MT, GATED, AHEAD>), hipFuncAttributeMaxDynamicSharedMemorySize, 8 * NT * MT * 4096));
        sized = true;
    }
    const dim3 grid(tiles, (row_tiles + MT - 1u) / MT, p.slices);
    hipLaunchKernelGGL((gemm_few_kernel<ELEMENT, MT, GATED, AHEAD>), grid, dim3(64u * p.deep), lds, d->stream, p);
    NH_HIP(hipGetLastError());
    return NH_OK;
}

template <int ELEMENT>
int32_t launch_element(nh_device *d, const FewParams &p, bool gated) {
    if (gated) return launch_few<ELEMENT, 1, true>(d, p);
    switch (few_row_tiles(p.N, p.rows, (uint32_t)d->compute_units)) {
        case 1: return launch_few<ELEMENT, 1, false>(d, p);
        case 2: return launch_few<ELEMENT, 2, false>(d, p);
        default: return launch_few<ELEMENT, 3, false>(d, p);
    }
}

}  // namespace

int gemm_few_held() {
    const char *held = getenv("NEURA_HIP_GEMM_FEW");
    return held && (held[0] == '0' || held[0] == '1') ? held[0] - '0' : -1;
}

bool gemm_few_takes(const nh_device *d, int32_t element, uint32_t N, uint32_t K, uint32_t rows) {
    if (const int held = gemm_few_held(); held >= 0) return held == 1;
    return few_rows_win(element, N, K, rows, (uint32_t)d->compute_units);
}

int32_t launch_gemm_few(nh_device *d, int32_t element, FewParams p, bool gated) {
    switch (element) {
        case NH_Q4_K: return launch_element<NH_Q4_K>(d, p, gated);
        case NH_Q5_K: return launch_element<NH_Q5_K>(d, p, gated);
        case NH_Q6_K: return launch_element<NH_Q6_K>(d, p, gated);
        case NH_Q3_K: return launch_element<NH_Q3_K>(d, p, gated);
        case NH_Q8_0: return launch_element<NH_Q8_0>(d, p, gated);
    }
    return fail(NH_E_ARGUMENT, "element %d carries no wide product", element);
}

}  // namespace nh
