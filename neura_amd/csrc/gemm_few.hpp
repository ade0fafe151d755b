// The wide product of few activation rows (gemm_few.hip), as the wide products' launcher (gemm.hip) reaches it.
#pragma once
#include "common.hpp"
#include "few_rule.hpp"

namespace nh {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t FEW_TILE = 32;  // weight rows and packed activation rows of a tile

// Where four neighbouring numbers (k a multiple of 4) of packed row `row` lie, in halves, when the rows are packed as the
// operands of v_mfma_f32_32x32x16_f16: [row / 32][k / 64][depth 0..3][part 0..1][row % 32][8], the eight numbers at
// k = 64 step + 8 chunk being depth 2 (chunk / 4) + chunk % 2 of part (chunk / 2) % 2 -- a wave reads an operand as 1 KB in a row.
__host__ __device__ inline size_t few_operand_at(uint32_t row, uint32_t k, uint32_t K) {
    const uint32_t chunk = (k >> 3) & 7u, depth = 2u * (chunk >> 2) + (chunk & 1u), part = (chunk >> 1) & 1u;
    return (((((size_t)(row >> 5) * (K >> 6) + (k >> 6)) * 4u + depth) * 2u + part) * 32u + (row & 31u)) * 8u + (k & 4u);
}
// and where the eight sub-block sums (part 0) or their residues (part 1) of a super-block lie: [row / 32][super-block][part][row % 32][8]
__host__ __device__ inline size_t few_sums_at(uint32_t row, uint32_t sb, uint32_t nsb, uint32_t part) {
    return ((((size_t)(row >> 5) * nsb + sb) * 2u + part) * 32u + (row & 31u)) * 8u;
}

// Whole fp32 rows (GemmArgs::whole): three half rows each, ten activation rows to a tile (its last two rows are never looked at).
constexpr uint32_t WHOLE_PIECES = 3, WHOLE_TILE = 10;
__host__ __device__ inline uint32_t whole_row(uint32_t m) { return m / WHOLE_TILE * FEW_TILE + m % WHOLE_TILE * WHOLE_PIECES; }
__host__ __device__ inline uint32_t whole_rows(uint32_t M) { return whole_row(M - 1u) + WHOLE_PIECES; }
// What the packing leaves of such a row beside its pieces.  A number that those do not hold to its last bit (less than 2^-36 of the
// row's largest, an infinity, a NaN) is a zero there and is listed as it is; past WHOLE_LISTED in one of the WHOLE_PARTS shares of the
// row the whole of it is read from `outside` instead.
constexpr uint32_t WHOLE_PARTS = 8, WHOLE_LISTED = 16;
struct WholeRow {
    float unscale;
    uint32_t unused;
    uint8_t listed[WHOLE_PARTS];  // numbers of each share of the row that the pieces do not hold, 255 at most
    struct {
        uint32_t k;
        float value;
    } list[WHOLE_PARTS][WHOLE_LISTED];
};
static_assert(sizeof(WholeRow) % 16u == 0, "read 16 bytes at a time");

// where K is shared among workgroups: the most their sums may take, and the most places they may meet at
constexpr size_t FEW_PARTIAL_BYTES = 16u << 20;
constexpr uint32_t FEW_MEETS = 1024;

struct FewParams {
    const uint8_t *W, *W1, *W2;  // matrices stacked along N, column ends end0 and end1 (multiples of the tile); gated: gate and up, N columns each
    uint32_t end0, end1;
    uint32_t N, K, row_bytes;
    const _Float16 *A, *S;  // packed rows and sums, in operand order
    uint32_t rows;          // rows of A: `pieces` of every activation row
    float *Y;
    const float *residual;
    uint32_t ldy, M;
    uint32_t pieces;        // 1 (half activations), 2, or WHOLE_PIECES: the rows of an activation row, each weighed 2^11 less than the one before
    const float *unscale;   // [M], with two pieces
    const WholeRow *whole;  // [M], with three
    const float *outside;   // [M][K], with three: the rows as fp32 numbers
    uint32_t deep;          // the waves of a workgroup: shares of K
    uint32_t slices;        // workgroups (blockIdx.z) that share the K of the same tiles
    float *partial;         // FEW_PARTIAL_BYTES of scratch for their sums
    uint32_t *meets;        // FEW_MEETS words, zero between launches: workgroups of a place that have left their sums
    uint32_t chain;         // of shared rows: units after which sums leave the accumulators
    float *Y1;              // where not null, columns from end0 on go there, with the same ldy (Y's first: Y1[n - end0])
};

int gemm_few_held();  // NEURA_HIP_GEMM_FEW: 0 never, 1 wherever it can be, -1 by the rule on sizes
// whether the product of `rows` packed rows is this kernel's, and its launch (the rows are packed)
bool gemm_few_takes(const nh_device *d, int32_t element, uint32_t N, uint32_t K, uint32_t rows);
int32_t launch_gemm_few(nh_device *d, int32_t element, const FewParams &p, bool gated);
// the product of shared rows (gemm_wide.hip), over rows packed the same way
int32_t launch_gemm_wide(nh_device *d, int32_t element, const FewParams &p, SharedShape shape);

}  // namespace nh
