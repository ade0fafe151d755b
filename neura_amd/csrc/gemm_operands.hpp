// What a lane of the wide products holds of one column's super-block, and the B operands of v_mfma_f32_32x32x16_f16 it makes of it in
// its registers, for every block format: lane l32 + 32 part takes runs of 16 stored numbers at 32 i + 16 part of ITS column, which are
// the pieces the blocks are stored in.
#pragma once
#include "blocks.hpp"
#include "gemm_few.hpp"

namespace nh {

namespace {

typedef const __attribute__((address_space(1))) u32x4 *global_uint4;
typedef const __attribute__((address_space(1))) uint8_t *global_bytes;
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
    // the next block's runs take a run's place once its operands are made (refill), its header waits beside this one's (advance)
    static constexpr bool IN_PLACE = true;
    u32x4 header_ahead, fifth_ahead;
    // (block: where the unit's block of the wave's first column lies; offset: the lane's column from there, pieces: its 16-byte pieces)
    __device__ __forceinline__ void refill(int g, __amdgpu_buffer_rsrc_t weights, uint32_t block, uint32_t offset, uint32_t pieces) {
        if (g == 0) {
            header_ahead = __builtin_amdgcn_raw_buffer_load_b128(weights, offset, block, 0);
            if (FIFTH) fifth_ahead = __builtin_amdgcn_raw_buffer_load_b128(weights, pieces + 16u, block, 0);
        }
        runs[g] = __builtin_amdgcn_raw_buffer_load_b128(weights, pieces + (FIFTH ? 48u : 16u) + 32u * g, block, 0);
    }
    __device__ __forceinline__ void advance() {
        header = header_ahead;
        if (FIFTH) fifth = fifth_ahead;
    }
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
    static __device__ __forceinline__ uint32_t centred(const u32x4 &header, int high) {  // 0xff where a sub-block's codes are centred, of four sub-blocks
        const uint32_t minimums = high ? ((header.w >> 4) & 0x0f0f0f0fu) | ((header.z >> 2) & 0x30303030u) : header.z & 0x3f3f3f3fu;
        const uint32_t some = (minimums + 0x7f7f7f7fu) & 0x80808080u;
        return some | (some - (some >> 7));
    }
    __device__ __forceinline__ float scale() const { return (float)as_halves(header.x).x * 16384.0f; }  // operands are code * sc * 2^-14
    static __device__ __forceinline__ float floor_scale(const u32x4 &header) { return (float)as_halves(header.x).y * -64.0f; }  // the sums are packed / 64
    static __device__ __forceinline__ float centre_scale(const u32x4 &header) { return (float)as_halves(header.x).x * (64.0f * CENTRE); }
    // the eight minimums (`scales`: the eight scales where the codes are centred) as halves; k 8..15 meet the sums' residues * 2^11
    static __device__ __forceinline__ half8_t floors(const u32x4 &header, uint32_t part, bool scales) {
        const half2_t offset = {(_Float16)1024.0f, (_Float16)1024.0f};
        const uint32_t first = scales ? header.y : header.z, more = scales ? header.w : header.w >> 4;
        const uint32_t lo4 = first & 0x3f3f3f3fu & (scales ? centred(header, 0) : ~0u), hi4 = ((more & 0x0f0f0f0fu) | ((first >> 2) & 0x30303030u)) & (scales ? centred(header, 1) : ~0u);
        half2_t m[4] = {as_halves(__builtin_amdgcn_perm(0u, lo4, 0x0c010c00u) | 0x64006400u) - offset,
                        as_halves(__builtin_amdgcn_perm(0u, lo4, 0x0c030c02u) | 0x64006400u) - offset,
                        as_halves(__builtin_amdgcn_perm(0u, hi4, 0x0c010c00u) | 0x64006400u) - offset,
                        as_halves(__builtin_amdgcn_perm(0u, hi4, 0x0c030c02u) | 0x64006400u) - offset};
        const _Float16 down = part ? (_Float16)0.00048828125f : (_Float16)1.0f;
        const half2_t downs = {down, down};
        return __builtin_bit_cast(half8_t, u32x4{as_word(m[0] * downs), as_word(m[1] * downs), as_word(m[2] * downs), as_word(m[3] * downs)});
    }
    // The minimums, and what centring took off, in units of the operands: (CENTRE * sc - dmin / d * m) / 256, in two pieces, to meet the
    // sums (packed / 64) where the operands meet the activations: ratio() first, then merged() for either four sub-blocks.  The pieces
    // hold 22 bits of what the block's own minimums hold exactly.  Up to dmin / d = 64 that is no further from 64 bits than the tiles,
    // which take them off exactly (2-norm, 512 x 3584, 100 rows: 8 1.27e-7 / 1.68e-7, 30 1.20 / 1.20, 60 1.11 / 1.12); beyond it is
    // (200 1.23 / 1.16, 5000 1.32 / 1.18), and ratio() says false: the pieces are zero then and floors() serve the block.  (Weights that
    // change sign lie around half the largest code, 8 and 16; d may be zero.)
    float down, up;
    __device__ __forceinline__ bool ratio(const u32x4 &header) {
        const float d = (float)as_halves(header.x).x, dmin = (float)as_halves(header.x).y;
        const float inverse = __builtin_amdgcn_rcpf(d);
        const float near = dmin * inverse, ratio = dmin == 0.0f ? 0.0f : fmaf(fmaf(-near, d, dmin), inverse, near);
        const bool fits = fabsf(ratio) <= 64.0f;
        down = fits ? ratio * -0.00390625f : 0.0f, up = fits ? CENTRE * 0.00390625f : 0.0f;
        return fits;
    }
    __device__ __forceinline__ void merged(const u32x4 &header, uint32_t part, int four, half8_t &coarse, half8_t &fine) const {
        const float share = part ? 0.00048828125f : 1.0f;  // (k 8..15 meet the sums' residues * 2^11)
        const uint32_t m = four ? ((header.w >> 4) & 0x0f0f0f0fu) | ((header.z >> 2) & 0x30303030u) : header.z & 0x3f3f3f3fu;
        const uint32_t sc = (four ? (header.w & 0x0f0f0f0fu) | ((header.y >> 2) & 0x30303030u) : header.y & 0x3f3f3f3fu) & centred(header, four);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float v = fmaf(down, (float)((m >> (8 * j)) & 255u), up * (float)((sc >> (8 * j)) & 255u));
            const _Float16 high = (_Float16)v;
            coarse[4 * four + j] = (_Float16)((float)high * share), fine[4 * four + j] = (_Float16)((v - (float)high) * share);
        }
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
        const uint32_t some = sc & (centred(header, g >> 1) >> shift);
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
    static constexpr bool IN_PLACE = false;
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
    static constexpr bool IN_PLACE = false;
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
    static constexpr bool IN_PLACE = false;
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

}  // namespace

}  // namespace nh
