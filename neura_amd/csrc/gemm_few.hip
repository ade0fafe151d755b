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
#include "gemm_operands.hpp"

#include <cmath>
#include <cstdlib>

namespace nh {

namespace {

static_assert(FEW_MEETS_MOST == FEW_MEETS && FEW_SUMS_MOST == FEW_PARTIAL_BYTES, "what the split counts on");

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
                    const half8_t b = w[t].floors(w[t].header, part, false), c = w[t].floors(w[t].header, part, true);
                    const float floor_scale = w[t].floor_scale(w[t].header), centre_scale = w[t].centre_scale(w[t].header);
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
    // (a second matrix with outputs of its own: the up projection beside the gate's)
    float *const Y = p.Y1 && n0 >= p.end0 ? p.Y1 - p.end0 : p.Y;
    auto leave = [&](uint32_t m, uint32_t n, float value, float up) {
        if (m >= p.M) return;
        if (GATED) value = value * (1.0f / (1.0f + expf(-value))) * up;
        const size_t to = (size_t)m * p.ldy + n;
        Y[to] = p.residual ? p.residual[to] + value : value;
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

template <int ELEMENT, int MT, bool GATED>
int32_t launch_few(nh_device *d, FewParams p) {
    constexpr int STEPS = FewOf<ELEMENT>::type::STEPS;
    constexpr int NT = GATED ? 2 : 1;
    constexpr int AHEAD = MT * NT > 2 ? 1 : (STEPS < 4 || MT * NT > 1 ? 2 : 4);
    const uint32_t tiles = (p.N + FEW_TILE - 1u) / FEW_TILE, row_tiles = (p.rows + FEW_TILE - 1u) / FEW_TILE;
    const FewSplit split = few_split(ELEMENT, p.N, p.K, p.rows, MT, NT, (uint32_t)d->compute_units);
    p.deep = split.deep, p.slices = split.slices;
    const size_t lds = (size_t)p.deep * NT * MT * 4096u;
    static OnceADevice sized;
    NH_HIP(raise_lds(sized, d, reinterpret_cast<const void *>(gemm_few_kernel<ELEMENT, MT, GATED, AHEAD>), 8 * NT * MT * 4096));
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

int32_t launch_gemm_few(nh_device *d, int32_t element, const FewParams &p, bool gated) {
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
