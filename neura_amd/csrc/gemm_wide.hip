// The wide product whose workgroups share their activation rows: Y[m][n] = sum_k X[m][k] * W[n][k], for every block format.
//
// Four or eight waves stand side by side over 32 columns each and MT tiles of 32 packed rows.  The rows' operands (few_operand_at:
// a tile's 16 k are 1 KB in a row) go through LDS, which the product of few rows leaves out: there every wave reads them for itself,
// 48 KB a super-block of three row tiles for 4.5 KB of weights, behind the weights' own loads.  Here a thread copies its pieces
// of half a unit two halves ahead, one a region (16 k), into a ring of three; the waves meet once a half.  A lane unpacks the weights of
// ITS column in its registers, as there, for MT products each.
//
// What bounds it is the vector unit: an instruction takes it 5 cycles beside 33 of a matrix product, and a product comes with five to
// seven of them (unpacking over MT, weighing, a block's minimums).  Hence: MT as large as 256 registers allow (two waves a SIMD: one
// alone issues an instruction in 5 cycles and waits out each latency); minimums and centres as two more products of the same
// accumulators, in units of the operands, where products of their own took three instructions an output; 32-bit offsets from
// uniform buffer descriptors; the next region's operands made and read while this one's products run, matrix and vector
// instructions by turns.  A region of four products and 22 vector instructions takes 36 cycles a product with two waves a SIMD.
// At full occupancy the card's clock gives way (2.3 to 1.8 GHz): 37888 x 3584 at 1024 packed rows, Q4_K, 344 us with the packing over one
// matrix again and again = 810 TFLOP/s (the 128 x 128 tiles 406), 352 over matrices from HBM, 351 to 366 without it in a fill; at 128 rows 65
// (few rows 76, tiles 77), at 74 rows 50, and 58 from HBM (few rows 56 and 63); 2-norm from 64 bits 1.2e-7 (tiles 1.7e-7 and more: uncentred).
#include "gemm_operands.hpp"

#include <type_traits>

namespace nh {

namespace {

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const uint8_t *at, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(at), 0, bytes, 0x00020000); }

// WN: waves side by side, 32 columns each; MT: tiles of 32 packed rows a wave multiplies its unpacked weights by; CHAINED: sums leave the
// accumulators every p.chain units (a kernel of one chain is one of fewer registers).
template <int ELEMENT, int WN, int MT, bool CHAINED>
__global__ __launch_bounds__(64 * WN, 2) void gemm_wide_kernel(FewParams p, uint32_t column_tiles, uint32_t row_blocks) {
    typedef typename FewOf<ELEMENT>::type Weights;
    constexpr int STEPS = Weights::STEPS, PLANES = Weights::PLANES, CLOSED = Weights::CLOSED, HALF = STEPS / 2, REGIONS = 4 * HALF;
    constexpr bool FLOORS = Weights::FLOORS, BLOCKS = ELEMENT == NH_Q8_0;  // (Q8_0's sums are weighed a block of two regions)
    constexpr uint32_t TILE = HALF * 4096u, STAGE = MT * TILE, THREADS = 64u * WN, COPIES = STAGE / 16u / THREADS;
    static_assert(STAGE / 16u % THREADS == 0 && MT <= WN, "every thread copies as many pieces, a wave a row tile's sums");
    extern __shared__ __attribute__((aligned(16))) uint8_t wide_lds[];
    uint8_t *const sums_lds = wide_lds + 3u * STAGE;
    const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, part = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // a die takes an eighth of the workgroups, in the order of the column tiles: the row blocks of one, which read the same weights,
    // follow one another there, and no die has more than another
    const uint32_t workgroups = column_tiles * row_blocks, each_die = (workgroups + 7u) / 8u;
    const uint32_t own_number = (blockIdx.x & 7u) * each_die + (blockIdx.x >> 3);
    if (own_number >= workgroups) return;
    const uint32_t column_tile = own_number / row_blocks, row_block = own_number - column_tile * row_blocks;
    const uint32_t steps = p.K / 64u, units = (steps + STEPS - 1u) / STEPS, nsb = p.K / 256u;
    const uint32_t last_tile = (p.rows - 1u) >> 5, tile0 = row_block * MT;
    const uint32_t column0 = column_tile * (32u * WN) + 32u * wave, n0 = min(column0, (p.N - 1u) & ~31u);  // (a wave past the last column does the last ones again)

    // the wave's 32 columns lie in one matrix
    const uint8_t *const wbase = n0 < p.end0 ? p.W + (size_t)n0 * p.row_bytes : n0 < p.end1 ? p.W1 + (size_t)(n0 - p.end0) * p.row_bytes : p.W2 + (size_t)(n0 - p.end1) * p.row_bytes;
    const uint32_t woff = min(l32, p.N - 1u - n0) * p.row_bytes;
    // ---- staging: half a unit is MT runs of TILE bytes.  (buffer loads: a uniform descriptor and offset, and 32 bits a lane.)
    constexpr bool EVEN = TILE / 16u % THREADS == 0;  // the threads' pieces are parts of one tile, the same for all
    u32x4 held[COPIES], held_sums;
    uint32_t from[COPIES], tile_at[COPIES];
#pragma unroll
    for (uint32_t i = 0; i < COPIES; i++) {
        const uint32_t piece = THREADS * i + (EVEN ? 0u : threadIdx.x);
        const uint32_t place = min(piece / (TILE / 16u), last_tile - tile0) * (steps * 4096u) + (piece % (TILE / 16u)) * 16u;
        tile_at[i] = EVEN ? place : 0u, from[i] = EVEN ? threadIdx.x * 16u : place;
    }
    const uint32_t own_tiles = min((uint32_t)MT, last_tile + 1u - tile0);
    const __amdgpu_buffer_rsrc_t rows_at = buffer_of(reinterpret_cast<const uint8_t *>(p.A) + (size_t)tile0 * steps * 4096u, own_tiles * steps * 4096u),
                                 sums_at = buffer_of(reinterpret_cast<const uint8_t *>(p.S) + (size_t)tile0 * nsb * 1024u, own_tiles * nsb * 1024u),
                                 weights_at = buffer_of(wbase, min(32u, p.N - n0) * p.row_bytes);
    const uint32_t sums_from = min(threadIdx.x >> 6, own_tiles - 1u) * (nsb * 1024u) + lane * 16u;
    const uint32_t last_half = steps / HALF - 1u;  // (an odd last step's unit has one half: the last one again, which meets zeros)
    auto fetch_piece = [&](uint32_t half, uint32_t i) {
        half = min(half, last_half);
        if (i < COPIES) held[i] = __builtin_amdgcn_raw_buffer_load_b128(rows_at, from[i], half * TILE + tile_at[i], 0);
        else if (FLOORS) held_sums = __builtin_amdgcn_raw_buffer_load_b128(sums_at, sums_from, (half >> 1) * 1024u, 0);
    };
    auto put_piece = [&](uint32_t half, uint32_t to, uint32_t i) {
        if (i < COPIES) *reinterpret_cast<u32x4 *>(wide_lds + to + (threadIdx.x + THREADS * i) * 16u) = held[i];
        else if (FLOORS && (half & 1u) == 0u && (MT >= WN || threadIdx.x < MT * 64u)) *reinterpret_cast<u32x4 *>(sums_lds + ((half >> 1) & 1u) * (MT * 1024u) + threadIdx.x * 16u) = held_sums;
    };

    f32x16 acc[MT], tmp[MT], zero;
#pragma unroll
    for (int e = 0; e < 16; e++) zero[e] = 0.0f;
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = zero;
    Weights w, next;
    auto ready = [&](Weights &of, uint32_t unit) {
        if constexpr (ELEMENT == NH_Q8_0) of.ready(wbase + woff, unit, steps, part);
        else if constexpr (ELEMENT == NH_Q6_K || ELEMENT == NH_Q3_K) of.ready(wbase + woff, unit, part);
    };
    // phase k: everyone has left half k in LDS, nobody reads half k - 2 any more; half k + 1 goes there, half k + 2 is asked for
    uint32_t phase = 0, to = STAGE, at = 0;
#pragma unroll
    for (uint32_t i = 0; i <= COPIES; i++) fetch_piece(0, i);
    w.fetch(wbase + woff, 0, steps, part);
#pragma unroll
    for (uint32_t i = 0; i <= COPIES; i++) put_piece(0, 0, i), fetch_piece(1u, i);
    __syncthreads();
    bool unfit = false;  // a block whose minimums meet no sums among the products (ratio)
    half8_t a[2][MT], b[2][PLANES], coarse, fine, sums[MT];
    auto read_rows = [&](int into, int r) {
#pragma unroll
        for (int i = 0; i < MT; i++) a[into][i] = *reinterpret_cast<const half8_t *>(wide_lds + at + lane * 16u + i * TILE + r * 1024u);
    };
    auto read_sums = [&](uint32_t unit) {
#pragma unroll
        for (int i = 0; i < MT; i++) sums[i] = *reinterpret_cast<const half8_t *>(sums_lds + (unit & 1u) * (MT * 1024u) + i * 1024u + lane * 16u);
    };
    auto floors = [&](int i) {
        tmp[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[i], coarse, tmp[i], 0, 0, 0);
        tmp[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[i], fine, tmp[i], 0, 0, 0);
    };
    // Where a chain of `chain` units ends, its sums leave the accumulators.  (Rows of residues, 2^11 below the rows they belong to, stay
    // and run on.)  SPARE: so many of a tile's sixteen registers hold on.  Sums that find none go to the outputs' own place (or to
    // scratch, where that still holds the residuals), each lane the outputs it writes at the end (18944 x 3584 Q3_K at 200 packed
    // rows, two chains of seven units, against one: 83 60.6 -> 59.5 us, 84 64.5 -> 69.0; 512 half rows: 42 in registers 123.6, 83 through
    // memory 113.7 -> 129.4).  Kernels of one chain do without, in 20 to 40 registers fewer (18944 x 3584 Q4_K at 400 packed rows 43 111 ->
    // 108 us; 42, of which a compute unit then holds three workgroups, 118 -> 108).
    constexpr int SPARE = shared_rows_spare(ELEMENT, WN, MT);
    const uint32_t pieces = p.pieces;
    float whole[SPARE ? MT : 1][SPARE ? SPARE : 1] = {};
    auto keep = [&](auto each, bool first, bool leave) __attribute__((always_inline)) {
        constexpr int EACH = decltype(each)::value;  // every packed row, or every second
        if constexpr (SPARE * EACH >= 16) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int e = 0; e < 16 / EACH; e++) {
                    whole[i][e] += acc[i][EACH * e];
                    acc[i][EACH * e] = leave ? 0.0f : whole[i][e];
                }
            return;
        }
        uint32_t seat = lane, ldk = p.residual ? p.N : p.ldy;
        asm volatile("" : "+v"(seat), "+v"(ldk));  // (worked out here: kept from before the walk, places and addresses would take its registers)
        const uint32_t column = n0 + (seat & 31u), rows = column < p.N && column0 < p.N ? p.M : 0u, row0 = tile0 * 32u / EACH + 4u / EACH * (seat >> 5);
        float *const kept = (p.residual ? p.partial : p.Y1 && n0 >= p.end0 ? p.Y1 - p.end0 : p.Y) + column;
        // (what the chains before left comes in one round trip, of four tiles in two; a place's sums leave before the next one's address
        // is made)
        constexpr int TOGETHER = MT == 4 ? 2 : MT;
#pragma unroll
        for (int i0 = 0; i0 < MT; i0 += TOGETHER) {
            float was[TOGETHER][4][4 / EACH];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TOGETHER; i++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t m = row0 + (32 * (i0 + i) + 8 * q) / EACH;
#pragma unroll
                    for (int e = 0; e < 4 / EACH; e++) was[i][q][e] = !first && m + e < rows ? kept[(size_t)(m + e) * ldk] : 0.0f;
                }
#pragma unroll
            for (int i = 0; i < TOGETHER; i++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    __builtin_amdgcn_sched_barrier(0);
                    const uint32_t m = row0 + (32 * (i0 + i) + 8 * q) / EACH;
#pragma unroll
                    for (int e = 0; e < 4 / EACH; e++) {
                        const float sum = was[i][q][e] + acc[i0 + i][4 * q + EACH * e];
                        if (leave && m + e < rows) kept[(size_t)(m + e) * ldk] = sum;
                        acc[i0 + i][4 * q + EACH * e] = leave ? 0.0f : sum;
                    }
                }
        }
    };
    auto keep_rows = [&](bool first, bool leave) __attribute__((always_inline)) {
        if (pieces == 2u) keep(std::integral_constant<int, 2>(), first, leave);
        else keep(std::integral_constant<int, 1>(), first, leave);
    };
    uint32_t until = CHAINED ? p.chain : 0u;
    read_rows(0, 0);
    ready(w, 0);
    w.step(0);
    w.operand(0, 0, b[0]);
    for (uint32_t unit = 0; unit < units; unit++) {
        const uint32_t after = min(unit + 1u, units - 1u);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // a region: 16 k.  The operands of the next are made as this one's products run
            if (h == 0) __builtin_amdgcn_s_setprio(0);
            else __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int r = 0; r < REGIONS; r++) {
                const int g = h * HALF + r / 4, depth = r & 3, cur = r & 1, nxt = cur ^ 1;
                const bool last = r == REGIONS - 1, first = BLOCKS ? (depth & 1) == 0 : g % CLOSED == 0 && depth == 0, end = h == 1 && last;
                const bool close = BLOCKS ? (depth & 1) == 1 : (g + 1) % CLOSED == 0 && depth == 3;
                __builtin_amdgcn_sched_barrier(0);
                if (last) {
                    __syncthreads();
                    phase++;
                    at = at == 2u * STAGE ? 0u : at + STAGE;
                    to = to == 2u * STAGE ? 0u : to + STAGE;
                    __builtin_amdgcn_sched_barrier(0);
                }
                read_rows(nxt, last ? 0 : r + 1);
                if (FLOORS && end) read_sums(unit);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    tmp[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[cur][i], b[cur][0], first ? zero : tmp[i], 0, 0, 0);
                    if (PLANES > 1) tmp[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[cur][i], b[cur][PLANES - 1], tmp[i], 0, 0, 0);
                }
                // (the minimums last: what they outweigh, where they do, meets them once and not at every product)
                if constexpr (FLOORS) {
                    if (end) {
#pragma unroll
                        for (int i = 0; i < MT; i++) floors(i);
                    }
                }
                float scale;
                if constexpr (BLOCKS) scale = w.block_scale(2 * g + (depth >> 1));
                else scale = w.scale();
                if (end) {
                    if constexpr (Weights::IN_PLACE) w.advance();
                    else w = next, ready(w, after);
                }
                const int of = (g + (depth == 3)) % STEPS;
                if (depth == 3) w.step(of);
                w.operand(of, (depth + 1) & 3, b[nxt]);
                if constexpr (FLOORS) {
                    if (h == 1 && r == 4) unfit = !w.ratio(w.header);
                    if (h == 1 && (r == 5 || r == 6)) w.merged(w.header, part, r - 5, coarse, fine);
                }
                if (!last) {
#pragma unroll
                    for (uint32_t i = 0; i <= COPIES; i++)
                        if (i * (REGIONS - 1) / (COPIES + 1u) == (uint32_t)r) put_piece(phase + 1u, to, i), fetch_piece(phase + 2u, i);
                }
                if constexpr (Weights::IN_PLACE) {
                    if (depth == 2) w.refill(g, weights_at, after * Weights::BYTES, woff, woff + 16u * part);
                } else {
                    if (h == 0 && r == 1) next.fetch(wbase + woff, after, steps, part);
                }
                if (FLOORS && end) __builtin_amdgcn_sched_group_barrier(0x100, 2 * MT, 0);
                else __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
                for (int i = 0; i < (FLOORS && end ? MT * 3 : MT * PLANES); i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                }
                if (close) {
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int e = 0; e < 16; e++) acc[i][e] = fmaf(scale, tmp[i][e], acc[i][e]);
                        asm volatile("" : "+v"(acc[i]));  // (here, not behind the products below: their sums are these registers)
                    }
                }
            }
        }
        if constexpr (FLOORS) {
            if (__any(unfit)) {  // (few blocks: minimums and centres each in products of their own)
                const u32x4 closed = __builtin_amdgcn_raw_buffer_load_b128(weights_at, woff, unit * Weights::BYTES, 0);
                read_sums(unit);
                const half8_t low = Weights::floors(closed, part, false), centre = Weights::floors(closed, part, true);
                const float low_scale = unfit ? Weights::floor_scale(closed) : 0.0f, centre_scale = unfit ? Weights::centre_scale(closed) : 0.0f;
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const f32x16 lows = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[i], low, zero, 0, 0, 0);
                    const f32x16 centres = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[i], centre, zero, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][e] += fmaf(low_scale, lows[e], centre_scale * centres[e]);
                }
            }
        }
        if (CHAINED && unit + 1u == until && until < units) keep_rows(until == p.chain, true), until += p.chain;
    }
    __builtin_amdgcn_s_setprio(0);
    // (every scale before the first store, and a tile's residuals before its stores: the compiler cannot tell them from the outputs, and
    // a chain of loads behind stores is a memory latency each, 16 us a workgroup)
    float scales[MT][4][4];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) scales[i][q][e] = pieces == 2u ? p.unscale[min((tile0 + i) * 16u + 4u * q + 2u * part + e / 2, p.M - 1u)] : 1.0f;  // (halves are packed as they lie)
    if (CHAINED && p.chain < units) keep_rows(false, false);

    // ---- out: lane (l32, part) holds column l32 of a 32 x 32 block; register 4q + e is row 8q + 4 part + e
    const uint32_t n = n0 + l32;
    if (n >= p.N || column0 >= p.N) return;
    // (a second matrix with outputs of its own: the up projection beside the gate's)
    float *const Y = p.Y1 && n >= p.end0 ? p.Y1 + (n - p.end0) : p.Y + n;
    const float *const residual = p.residual ? p.residual + n : nullptr;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        float beside[4][4];
        const uint32_t row = (tile0 + i) * 32u + 4u * part;
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t m = pieces == 2u ? ((row + 8u * q) >> 1) + (e & 1) : row + 8u * q + e;
                beside[q][e] = residual ? residual[(size_t)min(m, p.M - 1u) * p.ldy] : 0.0f;
            }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (pieces == 2u && e > 1) continue;
                const uint32_t m = pieces == 2u ? ((row + 8u * q) >> 1) + e : row + 8u * q + e;
                const float value = pieces == 2u ? fmaf(acc[i][4 * q + (2 * e + 1) % 4], 0.00048828125f, acc[i][4 * q + (2 * e) % 4]) * scales[i][q][(2 * e) % 4] : acc[i][4 * q + e] * scales[i][q][e];
                if (m < p.M) Y[(size_t)m * p.ldy] = residual ? beside[q][e] + value : value;
            }
    }
}

template <int ELEMENT, int WN, int MT, bool CHAINED>
int32_t launch_chained(nh_device *d, const FewParams &p) {
    typedef typename FewOf<ELEMENT>::type Weights;
    constexpr size_t lds = MT * (3u * (Weights::STEPS / 2u) * 4096u + (Weights::FLOORS ? 2048u : 0u));
    static OnceADevice sized;
    NH_HIP(raise_lds(sized, d, reinterpret_cast<const void *>(gemm_wide_kernel<ELEMENT, WN, MT, CHAINED>), lds));
    const uint32_t column_tiles = (p.N + 32u * WN - 1u) / (32u * WN), row_blocks = ((p.rows + 31u) / 32u + MT - 1u) / MT;
    hipLaunchKernelGGL((gemm_wide_kernel<ELEMENT, WN, MT, CHAINED>), dim3((column_tiles * row_blocks + 7u) / 8u * 8u), dim3(64 * WN), lds, d->stream, p, column_tiles, row_blocks);
    NH_HIP(hipGetLastError());
    return NH_OK;
}

template <int ELEMENT, int WN, int MT>
int32_t launch_shape(nh_device *d, FewParams p) {
    // (beside residuals the chains' sums wait in scratch: more of them than that holds stay in one chain)
    const uint32_t compute_units = (uint32_t)d->compute_units;
    const uint64_t residuals = p.residual ? (uint64_t)p.M * p.N * sizeof(float) : 0u;
    p.chain = shared_rows_chain(ELEMENT, p.N, p.K, p.rows, compute_units);
    if (p.chain >= shared_rows_units(ELEMENT, p.K) || shared_rows_overflow(ELEMENT, p.N, p.K, p.rows, residuals, compute_units)) return launch_chained<ELEMENT, WN, MT, false>(d, p);
    return launch_chained<ELEMENT, WN, MT, true>(d, p);
}

// (eight waves copy a step of Q8_0 in whole pieces only for two row tiles and four; two planes of Q6_K leave no registers for four)
template <int ELEMENT>
int32_t launch_element(nh_device *d, const FewParams &p, SharedShape shape) {
    constexpr bool Q8 = ELEMENT == NH_Q8_0, Q6 = ELEMENT == NH_Q6_K;
    if (shape == SHARED_42) return launch_shape<ELEMENT, 4, 2>(d, p);
    if (shape == SHARED_43 || (Q8 && shape == SHARED_83)) return launch_shape<ELEMENT, 4, 3>(d, p);
    if constexpr (!Q8) {
        if (shape == SHARED_83 || Q6) return launch_shape<ELEMENT, 8, 3>(d, p);
    }
    if constexpr (!Q6) return launch_shape<ELEMENT, 8, 4>(d, p);
    return fail(NH_E_ARGUMENT, "no shape %d of the product of shared rows", (int)shape);
}

}  // namespace

int32_t launch_gemm_wide(nh_device *d, int32_t element, const FewParams &p, SharedShape shape) {
    switch (element) {
        case NH_Q4_K: return launch_element<NH_Q4_K>(d, p, shape);
        case NH_Q5_K: return launch_element<NH_Q5_K>(d, p, shape);
        case NH_Q6_K: return launch_element<NH_Q6_K>(d, p, shape);
        case NH_Q3_K: return launch_element<NH_Q3_K>(d, p, shape);
        case NH_Q8_0: return launch_element<NH_Q8_0>(d, p, shape);
    }
    return fail(NH_E_ARGUMENT, "element %d carries no wide product", element);
}

}  // namespace nh
