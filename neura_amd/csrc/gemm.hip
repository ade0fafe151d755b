// Wide products (prefill): Y[m][n] = sum_k X[m][k] * W[n][k], W in raw GGUF blocks.
//
// Tile 64 (m) x 64 (n) x 32 (k) per 256-thread workgroup.  The weight tile is dequantised
// into LDS once per k step (one Q8_0 block / one sub-block of a super-block format deep) and reused by all 64
// activation rows; each thread owns a 4 x 4 patch of the output in registers.
#include "blocks.hpp"
#include "common.hpp"
#include "few_rule.hpp"
#include "gemm_few.hpp"
#include "gemv_shared.hpp"

#include <cstdlib>

namespace nh {

constexpr int BM = 64, BN = 64, BK = 32;

template <int ELEMENT, bool X_HALF>
__global__ __launch_bounds__(256) void gemm_kernel(const uint8_t *__restrict__ W, uint32_t N, uint32_t K, uint32_t row_bytes,
                                                   const void *__restrict__ X, uint32_t M, float *Y, const float *residual,
                                                   uint32_t ldy) {
    __shared__ float xs[BK][BM + 4];
    __shared__ float ws[BK][BN + 4];
    const uint32_t tid = threadIdx.x;
    const uint32_t m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const uint32_t tx = tid % 16, ty = tid / 16;  // patch: rows m0 + ty*4.., columns n0 + tx*4..
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.0f;

    for (uint32_t k0 = 0; k0 < K; k0 += BK) {
        // stage X: 64 rows x 32 k, thread -> (row = tid / 4, 8 consecutive k)
        {
            uint32_t r = tid / 4, kk = (tid % 4) * 8;
            uint32_t m = m0 + r;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float value = 0.0f;
                if (m < M && k0 + kk + j < K) {
                    if (X_HALF)
                        value = half_to_float(static_cast<const uint16_t *>(X)[(size_t)m * K + k0 + kk + j]);
                    else
                        value = static_cast<const float *>(X)[(size_t)m * K + k0 + kk + j];
                }
                xs[kk + j][r] = value;
            }
        }
        // stage W: 64 rows x 32 k dequantised
        {
            uint32_t r = tid / 4, kk = (tid % 4) * 8;
            uint32_t n = n0 + r;
            const uint8_t *row = W + (size_t)(n < N ? n : 0) * row_bytes;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float value = 0.0f;
                if (n < N && k0 + kk + j < K) value = stored_element<ELEMENT>(row, k0 + kk + j);
                ws[kk + j][r] = value;
            }
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BK; kk++) {
            float4 a = *reinterpret_cast<const float4 *>(&xs[kk][ty * 4]);
            float4 b = *reinterpret_cast<const float4 *>(&ws[kk][tx * 4]);
            const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float value = acc[i][j];
            if (residual) value = residual[(size_t)m * ldy + n] + value;
            Y[(size_t)m * ldy + n] = value;
        }
    }
}

// ------------------------------------------------------------------- Q4_K on MFMA --------
//
// Workgroup tile: 128 activation rows x 128 weight rows, walked 64 k at a time (one 64-element
// group of a super-block = sub-blocks 2g and 2g+1).  The 256 threads unpack the weight tile into
// LDS as halves holding code * sc -- an integer below 1024, exact in half precision -- so the
// matrix cores multiply exact integers by half-precision activations and add in fp32; after the
// four groups of a super-block the 64 x 64 result of each wave is weighed by d in fp32 and
// added to the running sums, and one more MFMA of depth 16 over (minimum, sub-block activation
// sum) pairs, weighed by dmin, takes the minimums off:
//     y = sum_blocks  d * sum_s sc_s * sum_k q_k x_k  -  dmin * sum_s m_s * sum_k x_k
// which is the reference's value (crates/neura-kernel/src/dot.rs:328-350, matmul.rs:1083-1221)
// regrouped per sub-block.  fp32 activations enter as two half rows each (the value rounded to
// half and the rounding residue times 2^11, after a power-of-two row scale), so 22 bits of
// every activation take part; half activations enter as they are.
//
// A nibble masked in place in a 16-bit lane is the half subnormal code * 2^-24 (or 2^-20);
// one packed half multiply by sc * 2^10 (or 2^6) turns it into the normal half code*sc*2^-14.
//
// Everything that does not depend on the weights is done once per activation row by a kernel
// of its own (gemm_pack_rows_kernel): the halves in the element order the unpacked nibbles come
// out in, and the sub-block sums the minimums are weighed by, already cut into the operand of
// their MFMA.  The tile loop is left with copies for the activations and four instructions
// per eight weights, and stages step s + 1 into the other half of LDS while the matrix cores
// walk step s: one barrier per step.

constexpr int GT = 128;           // tile edge (rows of A' and rows of W)
constexpr int GK = 64;            // k per step
constexpr int GS = GK + 8;        // LDS row stride in halves: 144 B keeps 128-bit reads of 8 neighbouring rows on distinct banks

struct GemmQ4Params {
    const uint8_t *W;
    const uint8_t *W1, *W2;  // matrices stacked along N behind W: columns [end0, end1) and [end1, N); both ends are multiples of the tile
    uint32_t end0, end1;
    uint32_t N, K, row_bytes;
    const _Float16 *A;   // [rows][K] halves, every four k in the order 0, 2, 1, 3; with `split`, row 2m is the rounded value of
                         // activation row m and row 2m+1 its residue * 2^11
    const _Float16 *S;   // [rows][K / 256][16]: the eight sub-block sums / 64 of a super-block as halves, then their residues * 2^11
    uint32_t rows;       // rows of A
    float *Y, *Y1;       // Y1: where not null, columns from end0 on go there (the second matrix's first to Y1[0])
    const float *residual;
    uint32_t ldy, M;
    int32_t split;
    const float *unscale;  // [M] with split: undoes the row scale
};

__device__ __forceinline__ void fetch_parameters(const GemmQ4Params &p) {
    NH_FETCH(p.W, p.W1, p.W2, p.end0, p.end1, p.N, p.K, p.row_bytes, p.A, p.S, p.rows, p.Y, p.Y1, p.residual, p.ldy, p.M, p.split, p.unscale);
}

// where column n of a tile from n0 on lies: [n] (a tile lies in one matrix)
__device__ __forceinline__ float *outputs_of(const GemmQ4Params &p, uint32_t n0) { return p.Y1 && n0 >= p.end0 ? p.Y1 - p.end0 : p.Y; }

// A number (times its row's scale) as PIECES halves whose weights fall by 2^11: two hold 22 of an fp32 number's bits; three hold all 24
// of every number down to 2^-36 of the row's largest.  Returns what is left over.
template <int PIECES>
__device__ __forceinline__ float cut(float t, _Float16 (&pieces)[PIECES][4], int at) {
#pragma unroll
    for (int j = 0; j < PIECES; j++) {
        pieces[j][at] = (_Float16)t;
        t = (t - (float)pieces[j][at]) * 2048.0f;  // (exact)
    }
    return t;
}

// Four neighbouring numbers of a row, cut into PIECES, into as many packed rows from `row` on, and their share of the sub-block sums:
// eight neighbouring lanes hold the 32 numbers of a sub-block.  FEW: in the operand order of the product of few rows
// (few_operand_at), not row by row.
template <int PIECES, bool FEW>
__device__ __forceinline__ void pack_piece(const _Float16 (&pieces)[PIECES][4], uint32_t row, uint32_t k, uint32_t K, uint32_t nsb,
                                           _Float16 *__restrict__ A, _Float16 *__restrict__ S) {
    const size_t place = FEW ? few_operand_at(row, k, K) : (size_t)row * K + k;
    float sums[PIECES];
#pragma unroll
    for (int j = 0; j < PIECES; j++) {
        // the nibbles of four weight bytes unpack as bytes 0, 2, 1, 3; (the rows of an activation row are neighbours in a tile)
        *reinterpret_cast<half4_t *>(A + place + (size_t)j * (FEW ? 8u : K)) = half4_t{pieces[j][0], pieces[j][2], pieces[j][1], pieces[j][3]};
        // sums of the 32 halves of a sub-block: eight neighbouring lanes
        sums[j] = ((float)pieces[j][0] + (float)pieces[j][1]) + ((float)pieces[j][2] + (float)pieces[j][3]);
    }
    if (!S) return;  // (weights without minimums)
#pragma unroll
    for (int j = 0; j < PIECES; j++) {
        sums[j] += dpp<DPP_QUAD_XOR1>(sums[j]);
        sums[j] += dpp<DPP_QUAD_XOR2>(sums[j]);
        sums[j] += dpp<DPP_ROW_HALF_MIRROR>(sums[j]);  // (a quad's lanes hold the same sum: the mirrored lane's is the other quad's)
    }
    if ((threadIdx.x & 7u) == 0) {
        const uint32_t sb = k >> 8, slot = (k >> 5) & 7u;
        float left = 0.0f;
#pragma unroll
        for (int j = 0; j < PIECES; j++) {
            // (a sum of 32 is longer than 22 bits, and the minimums' part largely cancels: what a row's sum drops goes into the next's)
            const float v = j ? fmaf(sums[j], 0.015625f, left) : sums[j] * 0.015625f;
            const _Float16 h = (_Float16)v;
            const float rest = (v - (float)h) * 2048.0f;
            const _Float16 residue = (_Float16)rest;
            _Float16 *dst = S + (FEW ? few_sums_at(row + j, sb, nsb, 0) : ((size_t)(row + j) * nsb + sb) * 16u);
            dst[slot] = h;
            dst[(FEW ? 256u : 8u) + slot] = residue;
            left = rest - (float)residue;
        }
    }
}

// the bits of a number's magnitude; FINITE: zero for an infinity or a NaN
template <bool FINITE>
__device__ __forceinline__ uint32_t magnitude(float v) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
    return FINITE && bits >= 0x7f800000u ? 0u : bits;
}

// What a whole row's packing leaves (WholeRow), for share blockIdx.y of the row: cutting a row in three is most of the packing's work
// (some 40 operations a number), and a few rows leave the chip idle, so WHOLE_PARTS workgroups take one each -- every one of them
// having read and measured the whole row by itself, which costs no time (7B ffn_down, eight rows: one workgroup a row 8 us).
template <class Get>
__device__ __forceinline__ void pack_whole(Get get, uint32_t K, uint32_t nsb, float scale, float back, _Float16 *__restrict__ A, _Float16 *__restrict__ S, WholeRow *__restrict__ whole,
                                           float *__restrict__ outside, uint32_t &listed) {
    const uint32_t m = blockIdx.x, part = blockIdx.y;
    const uint32_t quads = K / 4u, share = ((quads + WHOLE_PARTS - 1u) / WHOLE_PARTS + 7u) / 8u * 8u, end = min((part + 1u) * share, quads);  // whole sub-blocks
    for (uint32_t quad = part * share + threadIdx.x; quad < end; quad += blockDim.x) {
        const float4 v = get(4u * quad);
        const float held[4] = {v.x, v.y, v.z, v.w};
        _Float16 pieces[WHOLE_PIECES][4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float left = cut(held[e] * scale, pieces, e);
            if (!(left == 0.0f) || (held[e] != 0.0f && held[e] * scale == 0.0f)) {
#pragma unroll
                for (uint32_t j = 0; j < WHOLE_PIECES; j++) pieces[j][e] = (_Float16)0.0f;
                const uint32_t at = atomicAdd(&listed, 1u);
                if (at < WHOLE_LISTED) whole[m].list[part][at].k = 4u * quad + e, whole[m].list[part][at].value = held[e];
            }
        }
        *reinterpret_cast<float4 *>(outside + (size_t)m * K + 4u * quad) = v;
        pack_piece<WHOLE_PIECES, true>(pieces, whole_row(m), 4u * quad, K, nsb, A, S);
    }
    __syncthreads();
    if (threadIdx.x == 0) whole[m].unscale = back, whole[m].listed[part] = (uint8_t)min(listed, 255u);  // (the scale: the same word from every share)
}

// One workgroup per activation row (whole ones: WHOLE_PARTS): the row as MFMA-ready halves (fp32 rows: in PIECES rows, and a scale).
// PRELUDE: what a row is before it is packed -- 0: X as it lies; 1: X normalised (rmsnorm_kernel's arithmetic, so the same
// fp32 numbers: thread t adds the squares of columns t, t + 256, ..., then a 256-wide tree); 2: silu(gate) * X as
// silu_mul_kernel forms it.  `aux` is the norm's weight vector or the gate rows.
constexpr int PACK_PLAIN = 0, PACK_NORM = 1, PACK_SWIGLU = 2;
template <int PIECES, int PRELUDE, bool FEW>
__global__ __launch_bounds__(256) void gemm_pack_rows_kernel(const void *__restrict__ X, uint32_t K, _Float16 *__restrict__ A,
                                                             _Float16 *__restrict__ S, float *__restrict__ unscale,
                                                             const float *__restrict__ aux, float eps, WholeRow *__restrict__ whole, float *__restrict__ outside) {
    constexpr bool HALF_IN = PIECES == 1, WHOLE = PIECES == WHOLE_PIECES;
    static_assert(!(HALF_IN && PRELUDE != PACK_PLAIN), "half rows are packed as they lie");
    __shared__ uint32_t wave_top[4], listed;
    __shared__ float red[256];
    const uint32_t m = blockIdx.x, tid = threadIdx.x;
    const uint32_t nsb = (K + 255u) / 256u;
    float scale = 1.0f, norm = 1.0f, back = 1.0f;
    if (PRELUDE == PACK_NORM) {
        const float *xr = static_cast<const float *>(X) + (size_t)m * K;
        float square = 0.0f;
        for (uint32_t c = tid; c < K; c += 256) square = __fadd_rn(square, __fmul_rn(xr[c], xr[c]));
        red[tid] = square;
        __syncthreads();
        for (uint32_t stride = 128; stride > 0; stride >>= 1) {
            if (tid < stride) red[tid] = __fadd_rn(red[tid], red[tid + stride]);
            __syncthreads();
        }
        norm = rms_scale_of(red[0], K, eps);
    }
    // four neighbouring numbers of the row as the packing sees them
    auto fetch = [&](uint32_t k) -> float4 {
        float4 v = *reinterpret_cast<const float4 *>(static_cast<const float *>(X) + (size_t)m * K + k);
        if (PRELUDE == PACK_NORM) {
            const float4 w = *reinterpret_cast<const float4 *>(aux + k);
            v.x = __fmul_rn(__fmul_rn(v.x, norm), w.x), v.y = __fmul_rn(__fmul_rn(v.y, norm), w.y);
            v.z = __fmul_rn(__fmul_rn(v.z, norm), w.z), v.w = __fmul_rn(__fmul_rn(v.w, norm), w.w);
        } else if (PRELUDE == PACK_SWIGLU) {
            const float4 g = *reinterpret_cast<const float4 *>(aux + (size_t)m * K + k);
            v.x = g.x * (1.0f / (1.0f + expf(-g.x))) * v.x, v.y = g.y * (1.0f / (1.0f + expf(-g.y))) * v.y;
            v.z = g.z * (1.0f / (1.0f + expf(-g.z))) * v.z, v.w = g.w * (1.0f / (1.0f + expf(-g.w))) * v.w;
        }
        return v;
    };
    if (!HALF_IN) {
        uint32_t top = 0;
        for (uint32_t k = tid * 4u; k < K; k += 1024u) {
            const float4 v = fetch(k);
            top = max(max(top, magnitude<WHOLE>(v.x)), magnitude<WHOLE>(v.y));
            top = max(max(top, magnitude<WHOLE>(v.z)), magnitude<WHOLE>(v.w));
        }
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, offset, 64));
        if ((tid & 63u) == 0) wave_top[tid >> 6] = top;
        if (WHOLE && tid == 0) listed = 0;
        __syncthreads();
        top = max(max(wave_top[0], wave_top[1]), max(wave_top[2], wave_top[3]));
        // a power of two that puts the largest magnitude in [2^13, 2^14)
        const uint32_t raw = top >> 23, exponent = min(max(raw, 27u), 254u);
        scale = __builtin_bit_cast(float, (267u - exponent) << 23);
        back = raw == 255u ? __builtin_bit_cast(float, 0x7fc00000u) : __builtin_bit_cast(float, (exponent - 13u) << 23);
        if (!WHOLE && tid == 0) unscale[m] = back;
    }
    if constexpr (WHOLE) {
        pack_whole(fetch, K, nsb, scale, back, A, S, whole, outside, listed);
        return;
    }
    for (uint32_t k = tid * 4u; k < K; k += 1024u) {
        _Float16 pieces[PIECES][4];
        if (HALF_IN) {
            const half4_t v = *reinterpret_cast<const half4_t *>(static_cast<const _Float16 *>(X) + (size_t)m * K + k);
#pragma unroll
            for (int e = 0; e < 4; e++) pieces[0][e] = v[e];
        } else {
            const float4 v = fetch(k);
            const float held[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4; e++) cut(held[e] * scale, pieces, e);
        }
        pack_piece<PIECES, FEW>(pieces, PIECES * m, k, K, nsb, A, S);
    }
}

// The same for fp32 rows, through LDS: the kernel above walks a row three times (the norm's squares, the largest magnitude,
// the packing) and meets every value as it arrives -- a memory round trip a value and walk, 22 in a row on a 3584-wide row
// with the norm, 37 on an 18944-wide gated one.  Here a row crosses memory once, four 16-byte loads a thread in flight at a
// time, and waits in LDS as the prelude left it: the squares are added from LDS in the same thread order, the packing reads
// LDS.  The same arithmetic on the same numbers: the packed rows are the kernel above's bit for bit.  K is a multiple of 4.
// THREADS: 256, or 1024 where the rows are too few to fill the chip -- the loads of a wide row are then all in flight at once.
template <int PIECES, int PRELUDE, bool FEW, uint32_t THREADS>
__global__ __launch_bounds__(THREADS) void gemm_pack_rows_staged_kernel(const float *__restrict__ X, uint32_t K, _Float16 *__restrict__ A,
                                                                    _Float16 *__restrict__ S, float *__restrict__ unscale,
                                                                    const float *__restrict__ aux, float eps, WholeRow *__restrict__ whole, float *__restrict__ outside) {
    constexpr bool WHOLE = PIECES == WHOLE_PIECES;
    extern __shared__ __attribute__((aligned(16))) float staged_row[];  // [K]
    __shared__ uint32_t wave_top[THREADS / 64u], listed;
    __shared__ float red[256];
    const uint32_t m = blockIdx.x, tid = threadIdx.x;
    const uint32_t nsb = (K + 255u) / 256u;
    const float *xr = X + (size_t)m * K;
    const float *other = PRELUDE == PACK_NORM ? aux : (PRELUDE == PACK_SWIGLU ? aux + (size_t)m * K : nullptr);
    float norm = 1.0f;
    if (PRELUDE == PACK_NORM) {
        for (uint32_t k0 = tid * 4u; k0 < K; k0 += 16u * THREADS) {
            float4 held[4];
#pragma unroll
            for (int j = 0; j < 4; j++) held[j] = *reinterpret_cast<const float4 *>(xr + min(k0 + 4u * THREADS * j, K - 4u));
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (k0 + 4u * THREADS * j < K) *reinterpret_cast<float4 *>(staged_row + k0 + 4u * THREADS * j) = held[j];
        }
        __syncthreads();
        // thread t of the first 256 adds the squares of columns t, t + 256, ... as rmsnorm_kernel does, and so does the tree above them
        // (its last six levels within a wave)
        if (THREADS == 256u || tid < 256u) {
            float square = 0.0f;
            for (uint32_t c = tid; c < K; c += 256) square = __fadd_rn(square, __fmul_rn(staged_row[c], staged_row[c]));
            red[tid] = square;
        }
        __syncthreads();
        if (tid < 128u) red[tid] = __fadd_rn(red[tid], red[tid + 128u]);
        __syncthreads();
        if (tid < 64u) {
            float square = __fadd_rn(red[tid], red[tid + 64u]);
#pragma unroll
            for (int stride = 32; stride > 0; stride >>= 1) square = __fadd_rn(square, __shfl_down(square, stride, 64));
            if (tid == 0) red[0] = square;
        }
        __syncthreads();
        norm = rms_scale_of(red[0], K, eps);
    }
    uint32_t top = 0;
    for (uint32_t k0 = tid * 4u; k0 < K; k0 += 16u * THREADS) {
        float4 held[4], with[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t k = min(k0 + 4u * THREADS * j, K - 4u);
            held[j] = PRELUDE == PACK_NORM ? *reinterpret_cast<const float4 *>(staged_row + k) : *reinterpret_cast<const float4 *>(xr + k);
            if (PRELUDE != PACK_PLAIN) with[j] = *reinterpret_cast<const float4 *>(other + k);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (k0 + 4u * THREADS * j >= K) continue;
            float4 v = held[j];
            if (PRELUDE == PACK_NORM) {
                const float4 w = with[j];
                v.x = __fmul_rn(__fmul_rn(v.x, norm), w.x), v.y = __fmul_rn(__fmul_rn(v.y, norm), w.y);
                v.z = __fmul_rn(__fmul_rn(v.z, norm), w.z), v.w = __fmul_rn(__fmul_rn(v.w, norm), w.w);
            } else if (PRELUDE == PACK_SWIGLU) {
                const float4 g = with[j];
                v.x = g.x * (1.0f / (1.0f + expf(-g.x))) * v.x, v.y = g.y * (1.0f / (1.0f + expf(-g.y))) * v.y;
                v.z = g.z * (1.0f / (1.0f + expf(-g.z))) * v.z, v.w = g.w * (1.0f / (1.0f + expf(-g.w))) * v.w;
            }
            top = max(max(top, magnitude<WHOLE>(v.x)), magnitude<WHOLE>(v.y));
            top = max(max(top, magnitude<WHOLE>(v.z)), magnitude<WHOLE>(v.w));
            *reinterpret_cast<float4 *>(staged_row + k0 + 4u * THREADS * j) = v;  // the thread that packs these four wrote them
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, offset, 64));
    if ((tid & 63u) == 0) wave_top[tid >> 6] = top;
    if (WHOLE && tid == 0) listed = 0;
    __syncthreads();
    top = wave_top[0];
#pragma unroll
    for (uint32_t w = 1; w < THREADS / 64u; w++) top = max(top, wave_top[w]);
    // a power of two that puts the largest magnitude in [2^13, 2^14)
    const uint32_t raw = top >> 23, exponent = min(max(raw, 27u), 254u);
    const float scale = __builtin_bit_cast(float, (267u - exponent) << 23);
    const float back = raw == 255u ? __builtin_bit_cast(float, 0x7fc00000u) : __builtin_bit_cast(float, (exponent - 13u) << 23);
    if constexpr (WHOLE) {
        // (the share's numbers may be other threads': the barrier behind wave_top stands between)
        pack_whole([&](uint32_t k) { return *reinterpret_cast<const float4 *>(staged_row + k); }, K, nsb, scale, back, A, S, whole, outside, listed);
        return;
    }
    if (tid == 0) unscale[m] = back;
    for (uint32_t k = tid * 4u; k < K; k += 4u * THREADS) {
        const float4 v = *reinterpret_cast<const float4 *>(staged_row + k);
        const float held[4] = {v.x, v.y, v.z, v.w};
        _Float16 pieces[PIECES][4];
#pragma unroll
        for (int e = 0; e < 4; e++) cut(held[e] * scale, pieces, e);
        pack_piece<PIECES, FEW>(pieces, PIECES * m, k, K, nsb, A, S);
    }
}

static bool pack_unstaged() {  // NEURA_HIP_PACK_STAGED=0: the packing that walks a row in memory
    const char *held = getenv("NEURA_HIP_PACK_STAGED");
    return held && held[0] == '0';
}
constexpr size_t PACK_STAGED_LDS_MOST = 152 * 1024;  // the widest row the staged packing holds: 38912 numbers
constexpr size_t GEMM_Q4K_LDS = sizeof(_Float16) * (2 * GT * GS + 2 * GT * GS + 2 * GT * 8) + sizeof(uint32_t) * 2 * GT;

// What the multiplier waves of a super-block wide product do (waves 0..3 of the workgroup; the stagers fill As, Bs, mns and dds).
// The minimums (Q4_K, Q5_K) are taken off with one more MFMA per four steps over (minimum, activation sum) pairs;
// unscale_weights undoes the power of two the weights' operand was staged with.  Four steps share one (d, dmin) in dds[(step / 4) & 1].
__device__ __forceinline__ void gemm_multiply(const GemmQ4Params &p, _Float16 (*As)[GT][GS], _Float16 (*Bs)[GT][GS], _Float16 (*mns)[GT][8], uint32_t (*dds)[GT],
                                              const uint32_t wave, const uint32_t lane, const uint32_t n0, const uint32_t m0, const uint32_t steps, const float unscale_weights) {
    typedef const __attribute__((address_space(1))) u32x4 *global_uint4;
    // ---------------------------------------------------------------------- multipliers
    // wave (wm, wn) owns rows 64 wm.. of A' and weight rows 64 wn..
    const uint32_t wm = wave >> 1, wn = wave & 1u, l32 = lane & 31u, part = lane >> 5;
    const uint32_t nsb = p.K / 256u;
    const _Float16 *sums[2];
#pragma unroll
    for (int i = 0; i < 2; i++) sums[i] = p.S + (size_t)min(m0 + 64u * wm + 32u * i + l32, p.rows - 1u) * nsb * 16u + 8u * part;

    f32x16 acc[2][2], tmp[2][2], zero;
#pragma unroll
    for (int e = 0; e < 16; e++) zero[e] = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = zero, tmp[i][j] = zero;

    for (uint32_t first = 0; first < steps; first += 4) {
        const uint32_t sbuf = (first >> 2) & 1u;
        u32x4 sraw[2];
#pragma unroll
        for (int i = 0; i < 2; i++) sraw[i] = *(global_uint4)(uintptr_t)(sums[i] + (size_t)(first >> 2) * 16u);  // wanted at the end of the super-block
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t buf = g & 1u;
            __syncthreads();  // the step is staged
            // ---- 64 x 64 x 64 per wave; the operands of the next 16 k are on their way while the matrix cores walk these
            half8_t a[2][2], b[2][2];
            auto operands = [&](int kk) {
#pragma unroll
                for (int i = 0; i < 2; i++) a[kk & 1][i] = *reinterpret_cast<const half8_t *>(&As[buf][64u * wm + 32u * i + l32][16u * kk + 8u * part]);
#pragma unroll
                for (int j = 0; j < 2; j++) b[kk & 1][j] = *reinterpret_cast<const half8_t *>(&Bs[buf][64u * wn + 32u * j + l32][16u * kk + 8u * part]);
            };
            operands(0);
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                if (kk < 3) operands(kk + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        tmp[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[kk & 1][i], b[kk & 1][j], (g == 0 && kk == 0) ? zero : tmp[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- the super-block is complete: weigh by d, then take the minimums off
        float dscale[2], mscale[2];
        half8_t b2[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const half2_t dd = __builtin_bit_cast(half2_t, dds[sbuf][64u * wn + 32u * j + l32]);
            dscale[j] = (float)dd.x * unscale_weights;
            mscale[j] = (float)dd.y * -64.0f;  // the sums were packed / 64
            b2[j] = *reinterpret_cast<const half8_t *>(mns[sbuf][64u * wn + 32u * j + l32]);
            if (part) b2[j] = b2[j] * (_Float16)0.00048828125f;  // k 8..15: the minimums * 2^-11 against the residues * 2^11
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const half8_t a2 = __builtin_bit_cast(half8_t, sraw[i]);  // k 0..7: the sums; k 8..15: their residues
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = fmaf(dscale[j], tmp[i][j][e], acc[i][j][e]);
                const f32x16 mins = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2, b2[j], zero, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = fmaf(mscale[j], mins[e], acc[i][j][e]);
            }
        }
    }
    // ---- out: lane (l32, part) holds column n = l32 of a 32 x 32 block; register 4q + e is row 8q + 4 part + e
    float *const Y = outputs_of(p, n0);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t n = n0 + 64u * wn + 32u * j + l32;
            if (n >= p.N) continue;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t row = m0 + 64u * wm + 32u * i + 8u * q + 4u * part;  // first of four rows of A'
                if (p.split) {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const uint32_t m = (row >> 1) + e;
                        if (m >= p.M) continue;
                        float value = fmaf(acc[i][j][4 * q + 2 * e + 1], 0.00048828125f, acc[i][j][4 * q + 2 * e]) * p.unscale[m];
                        const size_t at = (size_t)m * p.ldy + n;
                        Y[at] = p.residual ? p.residual[at] + value : value;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t m = row + e;
                        if (m >= p.M) continue;
                        const size_t at = (size_t)m * p.ldy + n;
                        Y[at] = p.residual ? p.residual[at] + acc[i][j][4 * q + e] : acc[i][j][4 * q + e];
                    }
                }
            }
        }
}

// The eight waves of a workgroup split the work by kind.  Waves 4..7 (the stagers) fetch raw blocks and packed
// activations four steps ahead into registers, unpack step s + 1 into LDS; waves 0..3 (the multipliers) do nothing
// but read operands and drive the matrix cores over step s.  One stager and one multiplier share each SIMD, so
// unpacking and memory latency hide behind the MFMAs instead of taking turns with them.
//
// FIFTH: Q5_K.  The header is Q4_K's; behind it come 32 bytes of fifth bits (bit 2g of byte l belongs to weight l of group g's
// low half, bit 2g + 1 to weight 32 + l) and then the nibbles.  A code of five bits times a scale of six stays below 2048, so
// the operand is as exact as Q4_K's: the fifth bit is set beside the nibble before the one multiplication.
template <bool FIFTH>
__device__ __forceinline__ void gemm_q45k_mfma(const GemmQ4Params &p) {
    constexpr uint32_t BLOCK = FIFTH ? 176u : 144u, NIBBLES = FIFTH ? 48u : 16u;
    extern __shared__ __attribute__((aligned(16))) uint8_t gemm_lds[];
    _Float16(*As)[GT][GS] = reinterpret_cast<_Float16(*)[GT][GS]>(gemm_lds);                                           // [2]
    _Float16(*Bs)[GT][GS] = reinterpret_cast<_Float16(*)[GT][GS]>(gemm_lds + sizeof(_Float16) * 2 * GT * GS);          // [2]
    _Float16(*mns)[GT][8] = reinterpret_cast<_Float16(*)[GT][8]>(gemm_lds + sizeof(_Float16) * 4 * GT * GS);           // [2] by super-block parity: the eight minimums of every weight row
    uint32_t(*dds)[GT] = reinterpret_cast<uint32_t(*)[GT]>(gemm_lds + sizeof(_Float16) * (4 * GT * GS + 2 * GT * 8));  // [2]: (d, dmin) of every weight row
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n0 = blockIdx.x * GT, m0 = blockIdx.y * GT;
    const uint32_t steps = p.K / 64u;  // a multiple of 4: K is whole super-blocks
    typedef const __attribute__((address_space(1))) u32x4 *global_uint4;

    if (wave >= 4) {
        // ------------------------------------------------------------------ stagers
        // one row of each tile, one half (32 k) of the step
        const uint32_t tid = threadIdx.x - 256u;
        const uint32_t srow = tid >> 1, sh = tid & 1u;
        // a tile lies in one matrix: the boundaries between stacked matrices are multiples of the tile
        const uint32_t column = min(n0 + srow, p.N - 1u);
        const uint8_t *wrow = column < p.end0   ? p.W + (size_t)column * p.row_bytes
                              : column < p.end1 ? p.W1 + (size_t)(column - p.end0) * p.row_bytes
                                                : p.W2 + (size_t)(column - p.end1) * p.row_bytes;
        const _Float16 *arow = p.A + (size_t)min(m0 + srow, p.rows - 1u) * p.K + 32u * sh;
        u32x4 ahead, qs[4], av[4][4];  // the next super-block's header; groups and activations by slot = step % 4
        u32x4 fifth_ahead = {0u, 0u, 0u, 0u};  // Q5_K: the fifth bits of this thread's sixteen columns, next super-block
        const half2_t offset = {(_Float16)1024.0f, (_Float16)1024.0f}, powers = {(_Float16)1024.0f, (_Float16)64.0f};
        ahead = *(global_uint4)(uintptr_t)wrow;
        if (FIFTH) fifth_ahead = *(global_uint4)(uintptr_t)(wrow + 16u + 16u * sh);
#pragma unroll
        for (int g = 0; g < 4; g++) {  // steps 0..3 = super-block 0
            qs[g] = *(global_uint4)(uintptr_t)(wrow + NIBBLES + 32u * g + 16u * sh);
#pragma unroll
            for (int i = 0; i < 4; i++) av[g][i] = *(global_uint4)(uintptr_t)(arow + (size_t)g * 64u + 8 * i);
            __builtin_amdgcn_sched_barrier(0);  // slot 0 goes out first: the loop waits for the oldest slot only
        }
        for (uint32_t first = 0; first < steps; first += 4) {
            const u32x4 hdr = ahead, fifth = fifth_ahead;
            const uint32_t next = min((first >> 2) + 1u, (steps >> 2) - 1u);
            ahead = *(global_uint4)(uintptr_t)(wrow + (size_t)next * BLOCK);
            if (FIFTH) fifth_ahead = *(global_uint4)(uintptr_t)(wrow + (size_t)next * BLOCK + 16u + 16u * sh);
            const uint32_t fifth_words[4] = {fifth.x, fifth.y, fifth.z, fifth.w};
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint32_t buf = g & 1u, sbuf = (first >> 2) & 1u;
                // 6-bit fields of sub-blocks 2g, 2g+1 (crates/neura-precision/src/ggml.rs:127-136); 0x6400 | v is the half 1024 + v
                const uint32_t shift = 16u * (g & 1u);
                const uint32_t ya = (hdr.y >> shift) & 0xffffu, wa = (hdr.w >> shift) & 0xffffu;
                const uint32_t sc = g < 2 ? (ya & 0x3f3fu) : ((wa & 0x0f0fu) | ((ya >> 2) & 0x3030u));
                const uint32_t both = __builtin_amdgcn_perm(0u, sc, 0x0c010c00u) | 0x64006400u;  // (1024 + sc0, 1024 + sc1)
                const half2_t scales = (__builtin_bit_cast(half2_t, both) - offset) * powers;     // (sc0 * 2^10, sc1 * 2^6)
                const half2_t low_scale = {scales.x, scales.x}, high_scale = {scales.y, scales.y};
                const uint32_t words[4] = {qs[g].x, qs[g].y, qs[g].z, qs[g].w};
                uint32_t low[8], high[8];
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    const uint32_t even = words[w], odd = words[w] >> 8;
                    // element order inside a word: 0, 2 then 1, 3 (the byte lanes); the activations were packed in the same order
                    uint32_t low_even = even & 0x000f000fu, low_odd = odd & 0x000f000fu, high_even = even & 0x00f000f0u, high_odd = odd & 0x00f000f0u;
                    if (FIFTH) {
                        // bit 2g of a byte to bit 4 of its lane (beside the low nibble), bit 2g + 1 to bit 8 (beside the high nibble's four)
                        const uint32_t bits = fifth_words[w] >> (2 * g);
                        low_even |= (bits & 0x00010001u) << 4, low_odd |= ((bits >> 8) & 0x00010001u) << 4;
                        high_even |= (bits & 0x00020002u) << 7, high_odd |= ((bits >> 8) & 0x00020002u) << 7;
                    }
                    low[2 * w] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, low_even) * low_scale);
                    low[2 * w + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, low_odd) * low_scale);
                    high[2 * w] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, high_even) * high_scale);
                    high[2 * w + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, high_odd) * high_scale);
                }
                u32x4 *blow = reinterpret_cast<u32x4 *>(&Bs[buf][srow][16u * sh]), *bhigh = reinterpret_cast<u32x4 *>(&Bs[buf][srow][32u + 16u * sh]);
                blow[0] = u32x4{low[0], low[1], low[2], low[3]};
                blow[1] = u32x4{low[4], low[5], low[6], low[7]};
                bhigh[0] = u32x4{high[0], high[1], high[2], high[3]};
                bhigh[1] = u32x4{high[4], high[5], high[6], high[7]};
                if (g == 0 && sh == 0) {
                    // the eight minimums of the super-block, as halves
                    const uint32_t lo4 = hdr.z & 0x3f3f3f3fu;                                         // m0..m3
                    const uint32_t hi4 = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);  // m4..m7
                    const half2_t m01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, lo4, 0x0c010c00u) | 0x64006400u) - offset;
                    const half2_t m23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, lo4, 0x0c030c02u) | 0x64006400u) - offset;
                    const half2_t m45 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, hi4, 0x0c010c00u) | 0x64006400u) - offset;
                    const half2_t m67 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, hi4, 0x0c030c02u) | 0x64006400u) - offset;
                    *reinterpret_cast<u32x4 *>(mns[sbuf][srow]) = u32x4{__builtin_bit_cast(uint32_t, m01), __builtin_bit_cast(uint32_t, m23),
                                                                        __builtin_bit_cast(uint32_t, m45), __builtin_bit_cast(uint32_t, m67)};
                    dds[sbuf][srow] = hdr.x;
                }
                u32x4 *adst = reinterpret_cast<u32x4 *>(&As[buf][srow][32u * sh]);
#pragma unroll
                for (int i = 0; i < 4; i++) adst[i] = av[g][i];
                // the slot is free: the same group of the next super-block goes out.  Past the end the last super-block is
                // fetched again and dropped: with the same loads in every round the waits count exactly how many are newer
                {
                    const uint8_t *block = wrow + (size_t)next * BLOCK;
                    qs[g] = *(global_uint4)(uintptr_t)(block + NIBBLES + 32u * g + 16u * sh);
                    const _Float16 *at = arow + (size_t)(4u * next + g) * 64u;
#pragma unroll
                    for (int i = 0; i < 4; i++) av[g][i] = *(global_uint4)(uintptr_t)(at + 8 * i);
                }
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();  // step is staged; the multipliers are done with the step before it
            }
        }
        return;
    }

    gemm_multiply(p, As, Bs, mns, dds, wave, lane, n0, m0, steps, 16384.0f);  // the weights were staged * 2^-14
}

__global__ __launch_bounds__(512) void gemm_q4k_mfma_kernel(GemmQ4Params p) {
    fetch_parameters(p);
    gemm_q45k_mfma<false>(p);
}
__global__ __launch_bounds__(512) void gemm_q5k_mfma_kernel(GemmQ4Params p) {
    fetch_parameters(p);
    gemm_q45k_mfma<true>(p);
}

// ------------------------------------------------------------------- Q4_K, weights through registers --------
//
// LDS is what bounds the kernel above (it takes a workgroup's writes at 64 B a clock and serves its reads at 128: a step moves
// 32 KB in and 64 KB out, twice the time its MFMAs take).  Here the weights never touch it: eight multiplier waves own
// 64 x 32 of the 128 x 128 tile each, and lane (l32, part) of one loads, unpacks and feeds the matrix cores the weights of ITS
// row 32 wn + l32 -- per 64-k step one 16-byte load (bytes 16 part .. of the step's 32: the low nibbles are k = 16 part .. + 15,
// the high nibbles k = 32 + 16 part ..), whose four 8-weight pieces are the B operands of the step's four MFMA depths; the
// activation operand of depth kk is read from the matching 16-byte chunk of the staged row (chunk (kk >> 1) * 4 + 2 part +
// (kk & 1)), so the k order inside a step is the weights', not the natural one, and nothing has to move.  The header of a
// lane's row is in its registers, so d, dmin and the minimums need no LDS either.  Two multipliers share a SIMD (one unpacks
// while the other's MFMAs run) beside one of the four stagers, which only copy packed activation rows: whole 128-byte
// lines, eight lanes a row.  A stage of LDS is a whole super-block of k (256 columns of the 128 rows, 66 KB; two stages), so
// the twelve waves meet at one barrier a super-block, not one a step.
constexpr int GSB = 256 + 8;  // LDS row stride of a stage in halves: 528 B keeps 128-bit reads of 8 neighbouring rows on distinct banks
constexpr size_t GEMM_Q4K_REGB_LDS = sizeof(_Float16) * 2 * GT * GSB;

__global__ __launch_bounds__(768) void gemm_q4k_regb_mfma_kernel(GemmQ4Params p) {
    fetch_parameters(p);
    extern __shared__ __attribute__((aligned(16))) uint8_t gemm_lds[];
    _Float16(*As)[GT][GSB] = reinterpret_cast<_Float16(*)[GT][GSB]>(gemm_lds);  // [2]
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n0 = blockIdx.x * GT, m0 = blockIdx.y * GT;
    const uint32_t steps = p.K / 64u;  // a multiple of 4: K is whole super-blocks
    const uint32_t nsb = steps >> 2;
    typedef const __attribute__((address_space(1))) u32x4 *global_uint4;

    if (wave >= 8) {
        // ------------------------------------------------------------------ stagers: rows abase + 32 j, 16-byte chunks achunk + 8 c
        const uint32_t tid = threadIdx.x - 512u;
        const uint32_t abase = tid >> 3, achunk = tid & 7u;
        const _Float16 *asrc[4];
#pragma unroll
        for (int j = 0; j < 4; j++) asrc[j] = p.A + (size_t)min(m0 + abase + 32u * j, p.rows - 1u) * p.K + 8u * achunk;
        u32x4 av[4][4];  // the super-block on its way: [64-k step][row]
        auto fetch = [&](uint32_t sb) {
            const size_t at = (size_t)min(sb, nsb - 1u) * 256u;  // past the end the last super-block again, dropped
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int j = 0; j < 4; j++) av[c][j] = *(global_uint4)(uintptr_t)(asrc[j] + at + 64u * c);
        };
        fetch(0);
        for (uint32_t sb = 0; sb < nsb; sb++) {
            const uint32_t buf = sb & 1u;
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int j = 0; j < 4; j++) *reinterpret_cast<u32x4 *>(&As[buf][abase + 32u * j][64u * c + 8u * achunk]) = av[c][j];
            fetch(sb + 1u);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();  // the super-block is staged; the multipliers are done with the one before it
        }
        return;
    }

    // ---------------------------------------------------------------------- multipliers
    const uint32_t wm = wave >> 2, wn = wave & 3u, l32 = lane & 31u, part = lane >> 5;
    // a tile lies in one matrix: the boundaries between stacked matrices are multiples of the tile
    const uint32_t column = min(n0 + 32u * wn + l32, p.N - 1u);
    const uint8_t *wrow = column < p.end0   ? p.W + (size_t)column * p.row_bytes
                          : column < p.end1 ? p.W1 + (size_t)(column - p.end0) * p.row_bytes
                                            : p.W2 + (size_t)(column - p.end1) * p.row_bytes;
    const _Float16 *sums[2];
#pragma unroll
    for (int i = 0; i < 2; i++) sums[i] = p.S + (size_t)min(m0 + 64u * wm + 32u * i + l32, p.rows - 1u) * nsb * 16u + 8u * part;
    const half2_t offset = {(_Float16)1024.0f, (_Float16)1024.0f}, powers = {(_Float16)1024.0f, (_Float16)64.0f};

    f32x16 acc[2], tmp[2], zero;
#pragma unroll
    for (int e = 0; e < 16; e++) zero[e] = 0.0f;
    acc[0] = acc[1] = tmp[0] = tmp[1] = zero;

    // the lane's weights: a super-block's header and its four 16-byte runs, one super-block ahead
    u32x4 ahead, qs[4];
    ahead = *(global_uint4)(uintptr_t)wrow;
#pragma unroll
    for (int g = 0; g < 4; g++) qs[g] = *(global_uint4)(uintptr_t)(wrow + 16u + 32u * g + 16u * part);
    for (uint32_t first = 0; first < steps; first += 4) {
        const u32x4 hdr = ahead;
        const uint32_t next = min((first >> 2) + 1u, nsb - 1u);  // past the end the last super-block again, dropped
        ahead = *(global_uint4)(uintptr_t)(wrow + (size_t)next * 144u);
        u32x4 sraw[2];
#pragma unroll
        for (int i = 0; i < 2; i++) sraw[i] = *(global_uint4)(uintptr_t)(sums[i] + (size_t)(first >> 2) * 16u);  // wanted at the end of the super-block
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t sbuf = (first >> 2) & 1u;
            // 6-bit fields of sub-blocks 2g, 2g+1 (crates/neura-precision/src/ggml.rs:127-136); 0x6400 | v is the half 1024 + v
            const uint32_t shift = 16u * (g & 1u);
            const uint32_t ya = (hdr.y >> shift) & 0xffffu, wa = (hdr.w >> shift) & 0xffffu;
            const uint32_t sc = g < 2 ? (ya & 0x3f3fu) : ((wa & 0x0f0fu) | ((ya >> 2) & 0x3030u));
            const uint32_t both = __builtin_amdgcn_perm(0u, sc, 0x0c010c00u) | 0x64006400u;  // (1024 + sc0, 1024 + sc1)
            const half2_t scales = (__builtin_bit_cast(half2_t, both) - offset) * powers;     // (sc0 * 2^10, sc1 * 2^6)
            const half2_t low_scale = {scales.x, scales.x}, high_scale = {scales.y, scales.y};
            const uint32_t words[4] = {qs[g].x, qs[g].y, qs[g].z, qs[g].w};
            // the slot is free once its words are copied out: the same run of the next super-block goes out
            qs[g] = *(global_uint4)(uintptr_t)(wrow + (size_t)next * 144u + 16u + 32u * g + 16u * part);
            if (g == 0) __syncthreads();  // the super-block's activations are staged
            const _Float16 *arow0 = &As[sbuf][64u * wm + l32][64u * g], *arow1 = &As[sbuf][64u * wm + 32u + l32][64u * g];
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                // depth kk: words 2 (kk & 1), + 1 of the run, low nibbles for kk < 2; element order inside a word: 0, 2 then 1, 3
                // (the byte lanes), the order the activations were packed in
                uint32_t b[4];
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    const uint32_t even = words[2 * (kk & 1) + w], odd = even >> 8;
                    if (kk < 2) {
                        b[2 * w] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, even & 0x000f000fu) * low_scale);
                        b[2 * w + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, odd & 0x000f000fu) * low_scale);
                    } else {
                        b[2 * w] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, even & 0x00f000f0u) * high_scale);
                        b[2 * w + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, odd & 0x00f000f0u) * high_scale);
                    }
                }
                const half8_t weights = __builtin_bit_cast(half8_t, u32x4{b[0], b[1], b[2], b[3]});
                const uint32_t chunk = 8u * ((kk >> 1) * 4u + 2u * part + (kk & 1));  // where those eight k lie in the staged row
                const half8_t a0 = *reinterpret_cast<const half8_t *>(arow0 + chunk), a1 = *reinterpret_cast<const half8_t *>(arow1 + chunk);
                tmp[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, weights, (g == 0 && kk == 0) ? zero : tmp[0], 0, 0, 0);
                tmp[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, weights, (g == 0 && kk == 0) ? zero : tmp[1], 0, 0, 0);
            }
        }
        // ---- the super-block is complete: weigh by d, then take the minimums off (the eight minimums as halves, k 8..15 * 2^-11
        // against the sums' residues * 2^11)
        const half2_t dd = __builtin_bit_cast(half2_t, hdr.x);
        const float dscale = (float)dd.x * 16384.0f;  // the weights were unpacked * 2^-14
        const float mscale = (float)dd.y * -64.0f;    // the sums were packed / 64
        const uint32_t lo4 = hdr.z & 0x3f3f3f3fu;                                         // m0..m3
        const uint32_t hi4 = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);  // m4..m7
        half2_t m01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, lo4, 0x0c010c00u) | 0x64006400u) - offset;
        half2_t m23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, lo4, 0x0c030c02u) | 0x64006400u) - offset;
        half2_t m45 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, hi4, 0x0c010c00u) | 0x64006400u) - offset;
        half2_t m67 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, hi4, 0x0c030c02u) | 0x64006400u) - offset;
        if (part) {
            const half2_t down = {(_Float16)0.00048828125f, (_Float16)0.00048828125f};
            m01 = m01 * down, m23 = m23 * down, m45 = m45 * down, m67 = m67 * down;
        }
        const half8_t b2 = __builtin_bit_cast(half8_t, u32x4{__builtin_bit_cast(uint32_t, m01), __builtin_bit_cast(uint32_t, m23),
                                                             __builtin_bit_cast(uint32_t, m45), __builtin_bit_cast(uint32_t, m67)});
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const f32x16 mins = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, sraw[i]), b2, zero, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][e] = fmaf(dscale, tmp[i][e], acc[i][e]);
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][e] = fmaf(mscale, mins[e], acc[i][e]);
        }
    }
    // ---- out: lane (l32, part) holds column n = l32 of a 32 x 32 block; register 4q + e is row 8q + 4 part + e
    const uint32_t n = n0 + 32u * wn + l32;
    if (n >= p.N) return;
    float *const Y = outputs_of(p, n0);
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t row = m0 + 64u * wm + 32u * i + 8u * q + 4u * part;  // first of four rows of A'
            if (p.split) {
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const uint32_t m = (row >> 1) + e;
                    if (m >= p.M) continue;
                    float value = fmaf(acc[i][4 * q + 2 * e + 1], 0.00048828125f, acc[i][4 * q + 2 * e]) * p.unscale[m];
                    const size_t at = (size_t)m * p.ldy + n;
                    Y[at] = p.residual ? p.residual[at] + value : value;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t m = row + e;
                    if (m >= p.M) continue;
                    const size_t at = (size_t)m * p.ldy + n;
                    Y[at] = p.residual ? p.residual[at] + acc[i][4 * q + e] : acc[i][4 * q + e];
                }
            }
        }
    }
}

// ------------------------------------------------------------------- Q8_0 on MFMA --------
//
// The same tiles, the same packed activation rows and the same division of the waves.  A step of 64 k is two blocks: a
// stager owns one row and one block of the step, reads the nine words that cover its 34 bytes from the 4-byte boundary
// below it (a block starts on a half word as often as not; crates/neura-kernel/src/dot.rs:197-264 reads it the same way),
// and unpacks the 32 codes into LDS as the halves they are -- a signed byte b is the low byte of the half 1024 + 128 + b
// once its top bit is flipped, so one byte shuffle, one xor and one packed subtraction make two exact halves.  The block's
// scale cannot ride in the operand (a half times a byte is no half), so the multipliers close a sum after every block:
// two MFMAs of depth 16 into a fresh accumulator, then acc += d * sum in fp32 (run_weight_q8_0,
// crates/neura-kernel/src/task/matmul.rs:309-318, weighs a block the same way).  The weighing of one block runs on the
// vector unit while the matrix cores walk the next: the second block of a step is weighed behind the first MFMAs of the
// step after it.  K is a multiple of 64; steps are walked four at a time, the ones past the end as zero codes and zero
// scales, so every round issues the same loads and the waits count them exactly.
typedef uint32_t u32x4_loose __attribute__((ext_vector_type(4), aligned(4)));
constexpr size_t GEMM_Q8_LDS = sizeof(_Float16) * (4 * GT * GS) + sizeof(float) * 2 * 2 * GT;

__global__ __launch_bounds__(512) void gemm_q8_0_mfma_kernel(GemmQ4Params p) {
    fetch_parameters(p);
    extern __shared__ __attribute__((aligned(16))) uint8_t gemm_lds[];
    _Float16(*As)[GT][GS] = reinterpret_cast<_Float16(*)[GT][GS]>(gemm_lds);                                   // [2]
    _Float16(*Bs)[GT][GS] = reinterpret_cast<_Float16(*)[GT][GS]>(gemm_lds + sizeof(_Float16) * 2 * GT * GS);  // [2]
    float(*dds)[2][GT] = reinterpret_cast<float(*)[2][GT]>(gemm_lds + sizeof(_Float16) * 4 * GT * GS);         // [2][block of the step]: d of every weight row
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n0 = blockIdx.x * GT, m0 = blockIdx.y * GT;
    const uint32_t steps = p.K / 64u, walked = (steps + 3u) & ~3u;
    typedef const __attribute__((address_space(1))) u32x4 *global_uint4;
    typedef const __attribute__((address_space(1))) u32x4_loose *global_loose4;

    if (wave >= 4) {
        // ------------------------------------------------------------------ stagers
        const uint32_t tid = threadIdx.x - 256u;
        const uint32_t srow = tid >> 1, sh = tid & 1u;
        const uint32_t column = min(n0 + srow, p.N - 1u);
        const uint8_t *wrow = column < p.end0   ? p.W + (size_t)column * p.row_bytes
                              : column < p.end1 ? p.W1 + (size_t)(column - p.end0) * p.row_bytes
                                                : p.W2 + (size_t)(column - p.end1) * p.row_bytes;
        const _Float16 *arow = p.A + (size_t)min(m0 + srow, p.rows - 1u) * p.K + 32u * sh;
        u32x4 qa[4], qb[4], av[4][4];  // by slot = step % 4
        uint32_t qc[4];
        auto fetch = [&](int g, uint32_t step) {
            const uint32_t s = min(step, steps - 1u);  // past the end the last step is fetched again and dropped
            const uintptr_t at = (uintptr_t)(wrow + (size_t)(2u * s + sh) * 34u), low = at & ~(uintptr_t)3;
            qa[g] = *(global_loose4)low;
            qb[g] = *(global_loose4)(low + 16u);
            // a block on a word boundary ends two bytes into the ninth word: those two only are read (the last block of a
            // tensor ends where its allocation may)
            if (at & 2u) qc[g] = *(const __attribute__((address_space(1))) uint32_t *)(low + 32u);
            else qc[g] = *(const __attribute__((address_space(1))) uint16_t *)(low + 32u);
#pragma unroll
            for (int i = 0; i < 4; i++) av[g][i] = *(global_uint4)(uintptr_t)(arow + (size_t)s * 64u + 8 * i);
        };
#pragma unroll
        for (int g = 0; g < 4; g++) {
            fetch(g, (uint32_t)g);
            __builtin_amdgcn_sched_barrier(0);  // slot 0 goes out first: the loop waits for the oldest slot only
        }
        // (both walks start on a line of the instruction cache: where the length of what stands before left them, they took up to 5 %
        // longer -- 3584 x 18944 at 800 packed rows 250 us, here and where chance had them well 238)
        asm volatile(".p2align 6");
        const half2_t offset = {(_Float16)1152.0f, (_Float16)1152.0f};
        for (uint32_t first = 0; first < walked; first += 4) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint32_t buf = g & 1u, step = first + g;
                const bool odd = ((uintptr_t)(wrow + (size_t)(2u * min(step, steps - 1u) + sh) * 34u) & 2u) != 0;
                const uint32_t live = step < steps ? 0xffffffffu : 0u;
                const uint32_t words[9] = {qa[g].x, qa[g].y, qa[g].z, qa[g].w, qb[g].x, qb[g].y, qb[g].z, qb[g].w, qc[g]};
                const uint32_t scale_bits = (odd ? words[0] >> 16 : words[0] & 0xffffu) & live;
                uint32_t out[16];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t codes = (odd ? words[j + 1] : __funnelshift_r(words[j], words[j + 1], 16)) & live;
                    // element order inside a word: 0, 2 then 1, 3, the order the activations were packed in
                    const uint32_t even = __builtin_amdgcn_perm(0u, codes, 0x0c020c00u) ^ 0x64806480u;
                    const uint32_t uneven = __builtin_amdgcn_perm(0u, codes, 0x0c030c01u) ^ 0x64806480u;
                    out[2 * j] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, even) - offset);
                    out[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, uneven) - offset);
                }
                u32x4 *bdst = reinterpret_cast<u32x4 *>(&Bs[buf][srow][32u * sh]);
#pragma unroll
                for (int i = 0; i < 4; i++) bdst[i] = u32x4{out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]};
                dds[buf][sh][srow] = (float)__builtin_bit_cast(_Float16, (uint16_t)scale_bits);
                u32x4 *adst = reinterpret_cast<u32x4 *>(&As[buf][srow][32u * sh]);
#pragma unroll
                for (int i = 0; i < 4; i++) adst[i] = av[g][i];
                fetch(g, step + 4u);  // the slot is free: the same slot of the next round goes out
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();  // step is staged; the multipliers are done with the step before it
            }
        }
        return;
    }

    // ---------------------------------------------------------------------- multipliers
    const uint32_t wm = wave >> 1, wn = wave & 1u, l32 = lane & 31u, part = lane >> 5;
    f32x16 acc[2][2], tmp[2][2][2], zero;
#pragma unroll
    for (int e = 0; e < 16; e++) zero[e] = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = zero, tmp[0][i][j] = zero, tmp[1][i][j] = zero;
    float late[2] = {0.0f, 0.0f};  // the scales of the block whose sums wait in tmp[1]

    auto weigh = [&](int h, const float *scales) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = fmaf(scales[j], tmp[h][i][j][e], acc[i][j][e]);
    };

    asm volatile(".p2align 6");
    for (uint32_t step = 0; step < walked; step++) {
        const uint32_t buf = step & 1u;
        __syncthreads();  // the step is staged
        float early[2], next[2];
#pragma unroll
        for (int j = 0; j < 2; j++) early[j] = dds[buf][0][64u * wn + 32u * j + l32], next[j] = dds[buf][1][64u * wn + 32u * j + l32];
        half8_t a[2][2], b[2][2];
        auto operands = [&](int kk) {
#pragma unroll
            for (int i = 0; i < 2; i++) a[kk & 1][i] = *reinterpret_cast<const half8_t *>(&As[buf][64u * wm + 32u * i + l32][16u * kk + 8u * part]);
#pragma unroll
            for (int j = 0; j < 2; j++) b[kk & 1][j] = *reinterpret_cast<const half8_t *>(&Bs[buf][64u * wn + 32u * j + l32][16u * kk + 8u * part]);
        };
        operands(0);
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            if (kk < 3) operands(kk + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    tmp[kk >> 1][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[kk & 1][i], b[kk & 1][j], (kk & 1) ? tmp[kk >> 1][i][j] : zero, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // the sums the matrix cores are not writing are weighed meanwhile: the block before this step's first behind
            // its first MFMAs, this step's first behind the MFMAs of its second
            if (kk == 0) weigh(1, late);
            if (kk == 2) weigh(0, early);
            if (kk == 0 || kk == 2) __builtin_amdgcn_sched_barrier(0);
        }
        late[0] = next[0], late[1] = next[1];
    }
    weigh(1, late);
    // ---- out: lane (l32, part) holds column n = l32 of a 32 x 32 block; register 4q + e is row 8q + 4 part + e
    float *const Y = outputs_of(p, n0);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t n = n0 + 64u * wn + 32u * j + l32;
            if (n >= p.N) continue;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t row = m0 + 64u * wm + 32u * i + 8u * q + 4u * part;  // first of four rows of A'
                if (p.split) {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const uint32_t m = (row >> 1) + e;
                        if (m >= p.M) continue;
                        float value = fmaf(acc[i][j][4 * q + 2 * e + 1], 0.00048828125f, acc[i][j][4 * q + 2 * e]) * p.unscale[m];
                        const size_t at = (size_t)m * p.ldy + n;
                        Y[at] = p.residual ? p.residual[at] + value : value;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t m = row + e;
                        if (m >= p.M) continue;
                        const size_t at = (size_t)m * p.ldy + n;
                        Y[at] = p.residual ? p.residual[at] + acc[i][j][4 * q + e] : acc[i][j][4 * q + e];
                    }
                }
            }
        }
}

// Where a wide product's packed rows lie in the device's scratch: whole tiles of K halves a row, as many of [K / 256][16] sums, M row
// scales (whole rows: WholeRow, and the rows themselves), the sums workgroups of the product of few rows leave each other (the same for
// every product over the same rows: `packed` ones find them where they were).
struct PackedRows {
    size_t sums, unscale, outside, partial, bytes;
    PackedRows(uint32_t M, uint32_t K, uint32_t pieces) {
        const bool whole = pieces == WHOLE_PIECES;
        const size_t rows = ((whole ? (size_t)whole_rows(M) : (size_t)M * pieces) + FEW_TILE - 1u) / FEW_TILE * FEW_TILE;  // (whole tiles: few_operand_at)
        sums = rows * K * sizeof(_Float16);
        unscale = sums + rows * ((K + 255u) / 256u) * 16u * sizeof(_Float16);
        outside = unscale + ((size_t)M * (whole ? sizeof(WholeRow) : sizeof(float)) + 15u) / 16u * 16u;
        partial = outside + (whole ? (size_t)M * K * sizeof(float) : 0u);
        bytes = partial + FEW_PARTIAL_BYTES;
    }
};
size_t gemm_scratch_bytes(uint32_t M, uint32_t K, uint32_t pieces) { return PackedRows(M, K, pieces).bytes; }

template <int PIECES, int PRELUDE, bool FEW, uint32_t THREADS>
static int32_t pack_staged(nh_device *d, const GemmArgs &a, size_t lds, _Float16 *A, _Float16 *S, float *unscale, const float *aux, float *outside) {
    static OnceADevice roomy;
    NH_HIP(raise_lds(roomy, d, reinterpret_cast<const void *>(gemm_pack_rows_staged_kernel<PIECES, PRELUDE, FEW, THREADS>), PACK_STAGED_LDS_MOST));
    hipLaunchKernelGGL((gemm_pack_rows_staged_kernel<PIECES, PRELUDE, FEW, THREADS>), dim3(a.M, PIECES == WHOLE_PIECES ? WHOLE_PARTS : 1u), dim3(THREADS), lds, d->stream, static_cast<const float *>(a.X), a.K, A, S, unscale, aux, a.eps, reinterpret_cast<WholeRow *>(unscale), outside);
    NH_HIP(hipGetLastError());
    return NH_OK;
}

template <int PIECES, int PRELUDE, bool FEW>
static int32_t pack_fp32(nh_device *d, const GemmArgs &a, _Float16 *A, _Float16 *S, float *unscale, const float *aux, float *outside) {
    if (a.K % 4u == 0 && a.K >= 4u && (size_t)a.K * sizeof(float) <= PACK_STAGED_LDS_MOST && !pack_unstaged()) {
        // a row of fp32 numbers crosses memory once and waits in LDS
        const size_t lds = (size_t)a.K * sizeof(float);
        if (a.M > 2u * (uint32_t)d->compute_units) return pack_staged<PIECES, PRELUDE, FEW, 256>(d, a, lds, A, S, unscale, aux, outside);
        return pack_staged<PIECES, PRELUDE, FEW, 1024>(d, a, lds, A, S, unscale, aux, outside);
    }
    hipLaunchKernelGGL((gemm_pack_rows_kernel<PIECES, PRELUDE, FEW>), dim3(a.M, PIECES == WHOLE_PIECES ? WHOLE_PARTS : 1u), dim3(256), 0, d->stream, a.X, a.K, A, S, unscale, aux, a.eps,
                       reinterpret_cast<WholeRow *>(unscale), outside);
    NH_HIP(hipGetLastError());
    return NH_OK;
}

template <int PIECES, bool FEW>
static int32_t pack_rows(nh_device *d, const GemmArgs &a, _Float16 *A, _Float16 *S, float *unscale, float *outside) {
    const float *none = nullptr;
    if constexpr (PIECES == 1) {
        hipLaunchKernelGGL((gemm_pack_rows_kernel<1, PACK_PLAIN, FEW>), dim3(a.M), dim3(256), 0, d->stream, a.X, a.K, A, S, unscale, none, 0.0f, nullptr, outside);
        NH_HIP(hipGetLastError());
        return NH_OK;
    } else {
        if (a.norm_w) return pack_fp32<PIECES, PACK_NORM, FEW>(d, a, A, S, unscale, a.norm_w, outside);
        if (a.gate) return pack_fp32<PIECES, PACK_SWIGLU, FEW>(d, a, A, S, unscale, a.gate, outside);
        return pack_fp32<PIECES, PACK_PLAIN, FEW>(d, a, A, S, unscale, none, outside);
    }
}

// Which form a wide product takes.  `operands`: over rows packed in operand order (the product of few rows, or of shared rows in a
// shape), else the 128 x 128 tiles.  NEURA_HIP_GEMM_WIDE=0: no shared rows; =42, 43, 83, 84: that shape wherever it can.  Q6_K and
// Q3_K have no tiles: past the height of the product of few rows' grid, and where NEURA_HIP_GEMM_FEW=0 keeps them from it, they go to shared
// rows whatever is held.
struct WideForm {
    bool operands;
    SharedShape shape;
};
static WideForm wide_form(const nh_device *d, int32_t element, uint32_t N, uint32_t K, uint32_t rows, bool halves, size_t residuals) {
    // (`residuals`: bytes of outputs whose place holds residuals)
    const uint32_t units = (uint32_t)d->compute_units;
    const int held = shared_rows_overflow(element, N, K, rows, residuals, units) ? 0 : env_int("NEURA_HIP_GEMM_WIDE", -1);
    if (held == SHARED_42 || held == SHARED_43 || held == SHARED_83 || held == SHARED_84) return WideForm{true, (SharedShape)held};
    const SharedShape shape = held == 0 || gemm_few_held() >= 0 ? SHARED_NONE : shared_rows_shape(element, N, K, rows, halves, units);
    if (shape != SHARED_NONE || gemm_few_takes(d, element, N, K, rows)) return WideForm{true, shape};
    const bool tiled = element != NH_Q6_K && element != NH_Q3_K;
    return tiled ? WideForm{false, SHARED_NONE} : WideForm{true, SHARED_43};
}

static int32_t launch_gemm_mfma(nh_device *d, const GemmArgs &a) {
    GemmQ4Params p{};
    p.W = static_cast<const uint8_t *>(a.W);
    p.W1 = static_cast<const uint8_t *>(a.W_more[0]), p.W2 = static_cast<const uint8_t *>(a.W_more[1]);
    p.end0 = p.W1 ? a.end[0] : a.N, p.end1 = p.W2 ? a.end[1] : a.N;
    if ((p.W1 && (p.end0 % GT || p.end0 > a.N)) || (p.W2 && (!p.W1 || p.end1 % GT || p.end1 < p.end0 || p.end1 > a.N)))
        return fail(NH_E_ARGUMENT, "matrices stacked at columns %u and %u of %u do not fall on tiles of %d", a.end[0], a.end[1], a.N, GT);
    p.N = a.N;
    p.K = a.K;
    p.row_bytes = (uint32_t)payload_bytes(a.element, a.K);
    p.Y = a.Y, p.Y1 = a.Y_more;
    p.residual = a.residual;
    p.ldy = a.ldy;
    p.M = a.M;
    const bool half_rows = a.x_element == NH_F16;
    const uint32_t pieces = half_rows ? 1u : a.whole ? WHOLE_PIECES : 2u;
    p.rows = a.whole ? whole_rows(a.M) : pieces * a.M;
    p.split = half_rows ? 0 : 1;
    const WideForm form = a.whole || a.gated ? WideForm{true, SHARED_NONE} : wide_form(d, a.element, a.N, a.K, p.rows, half_rows, a.residual ? (size_t)a.M * a.N * sizeof(float) : 0u);
    const bool few = form.operands;
    if (a.whole && (half_rows || gemm_few_held() == 0 || a.M > 65535u * WHOLE_TILE))
        return fail(NH_E_ARGUMENT, "this wide product takes no fp32 rows whole (ask gemm_takes_whole first)");
    if (a.gated && (!gemm_few_takes(d, a.element, a.N, a.K, p.rows) || !p.W1 || p.W2 || a.residual || p.end0 != a.N))
        return fail(NH_E_ARGUMENT, "this wide product gates no outputs (ask gemm_gates first)");
    const PackedRows at(a.M, a.K, pieces);
    uint8_t *room = static_cast<uint8_t *>(scratch(d, at.bytes));
    if (!room) return NH_E_MEMORY;
    _Float16 *A = reinterpret_cast<_Float16 *>(room), *S = reinterpret_cast<_Float16 *>(room + at.sums);
    float *unscale = reinterpret_cast<float *>(room + at.unscale), *outside = reinterpret_cast<float *>(room + at.outside);
    if ((a.norm_w || a.gate) && (half_rows || (a.norm_w && a.gate) || ((uintptr_t)(a.norm_w ? a.norm_w : a.gate) & 15u)))
        return fail(NH_E_ARGUMENT, "a wide product normalises or gates fp32 rows read from 16-byte aligned addresses, one of the two");
    const bool sums = a.shared || a.element == NH_Q4_K || a.element == NH_Q5_K;  // whether weights with minimums meet these rows
    if (!a.packed) {  // (rows packed by the launch before are this launch's operand)
        const int32_t status = half_rows ? (few ? pack_rows<1, true>(d, a, A, S, unscale, outside) : pack_rows<1, false>(d, a, A, S, unscale, outside))
                               : a.whole ? pack_rows<WHOLE_PIECES, true>(d, a, A, sums ? S : nullptr, unscale, outside)
                               : few     ? pack_rows<2, true>(d, a, A, S, unscale, outside)
                                         : pack_rows<2, false>(d, a, A, S, unscale, outside);
        if (status != NH_OK) return status;
    }
    p.A = A, p.S = S, p.unscale = unscale;
    if (few) {
        const FewParams f{p.W, p.W1, p.W2, p.end0, p.end1, p.N, p.K, p.row_bytes, p.A, p.S, p.rows, p.Y, p.residual, p.ldy, p.M, pieces, p.unscale, reinterpret_cast<const WholeRow *>(unscale), outside,
                          1u, 1u, reinterpret_cast<float *>(room + at.partial), d->meets, 0u, a.Y_more};
        return form.shape != SHARED_NONE ? launch_gemm_wide(d, a.element, f, form.shape) : launch_gemm_few(d, a.element, f, a.gated);
    }
    static OnceADevice sized[4];
    NH_HIP(raise_lds(sized[0], d, reinterpret_cast<const void *>(gemm_q4k_mfma_kernel), GEMM_Q4K_LDS));
    NH_HIP(raise_lds(sized[1], d, reinterpret_cast<const void *>(gemm_q8_0_mfma_kernel), GEMM_Q8_LDS));
    NH_HIP(raise_lds(sized[2], d, reinterpret_cast<const void *>(gemm_q4k_regb_mfma_kernel), GEMM_Q4K_REGB_LDS));
    NH_HIP(raise_lds(sized[3], d, reinterpret_cast<const void *>(gemm_q5k_mfma_kernel), GEMM_Q4K_LDS));
    dim3 grid((a.N + GT - 1) / GT, (p.rows + GT - 1) / GT);
    if (a.element == NH_Q8_0) hipLaunchKernelGGL(gemm_q8_0_mfma_kernel, grid, dim3(512), GEMM_Q8_LDS, d->stream, p);
    else if (a.element == NH_Q5_K) hipLaunchKernelGGL(gemm_q5k_mfma_kernel, grid, dim3(512), GEMM_Q4K_LDS, d->stream, p);
    else if (const char *held = getenv("NEURA_HIP_GEMM_REGB"); held && held[0] == '0')  // the form that unpacks the weights into LDS
        hipLaunchKernelGGL(gemm_q4k_mfma_kernel, grid, dim3(512), GEMM_Q4K_LDS, d->stream, p);
    else hipLaunchKernelGGL(gemm_q4k_regb_mfma_kernel, grid, dim3(768), GEMM_Q4K_REGB_LDS, d->stream, p);
    NH_HIP(hipGetLastError());
    return NH_OK;
}

// the matrix-core forms take Q4_K, Q5_K, Q6_K and Q3_K rows of whole super-blocks and Q8_0 rows of whole pairs of blocks, read
// from 16-byte aligned addresses (a Q8_0, Q6_K or Q3_K matrix from a 4-byte one; its rows may start on any half word)
static bool mfma_takes(int32_t element, uint32_t K, const void *X, const void *W) {
    const char *held = getenv("NEURA_HIP_GEMM_MFMA");
    const bool wanted = !(held && held[0] == '0');
    const bool aligned = ((uintptr_t)X & 15u) == 0 && ((uintptr_t)W & (element == NH_Q4_K || element == NH_Q5_K ? 15u : 3u)) == 0;
    return wanted && aligned && K > 0 &&
           (((element == NH_Q4_K || element == NH_Q5_K || element == NH_Q6_K || element == NH_Q3_K) && K % 256u == 0) || (element == NH_Q8_0 && K % 64u == 0));
}

bool gemm_stacks(int32_t element, uint32_t K, const void *X, const void *W0, const void *W1, const void *W2, uint32_t end0, uint32_t end1) {
    if (!mfma_takes(element, K, X, W0)) return false;
    const uintptr_t loose = element == NH_Q4_K || element == NH_Q5_K ? 15u : 3u;
    if (W1 && (((uintptr_t)W1 & loose) || end0 % GT)) return false;
    if (W2 && (((uintptr_t)W2 & loose) || end1 % GT || !W1)) return false;
    return true;
}

bool gemm_takes_whole(int32_t element, uint32_t K, const void *X, const void *W) {
    return gemm_few_held() != 0 && mfma_takes(element, K, X, W);
}

// one launch for the gate and the up projection, silu(gate) * up leaving it: the product of few rows
bool gemm_gates(const nh_device *d, int32_t element, uint32_t N, uint32_t K, uint32_t rows, const void *X, const void *gate, const void *up) {
    return N % GT == 0 && gemm_stacks(element, K, X, gate, nullptr, nullptr, 0, 0) && gemm_stacks(element, K, X, up, nullptr, nullptr, 0, 0) &&
           rows <= FEW_TILE && gemm_few_takes(d, element, N, K, rows);
}

bool gemm_shares_rows(const nh_device *d, const int32_t (&elements)[3], const uint8_t *const (&W)[3], const uint32_t (&N)[3], uint32_t K, const void *X, uint32_t M, bool whole) {
    if (whole) {
        if (env_int("NEURA_HIP_GEMV_WIDE", 1) == 0) return false;  // one narrow product a matrix
        for (int s = 0; s < 3; s++)
            if (!gemm_takes_whole(elements[s], K, X, W[s])) return false;
        return true;
    }
    for (int s = 0; s < 3; s++)
        if (!mfma_takes(elements[s], K, X, W[s]) || wide_form(d, elements[s], N[s], K, 2u * M, false, 0u).operands != wide_form(d, elements[0], N[0], K, 2u * M, false, 0u).operands) return false;
    return true;
}

// (the rule's measurements are beside it; the error against 64 bits is no larger -- N(0, 1) rows, 2-norm, the decoder shapes: Q8_0
// 2.3..3.1e-7 -> 0.8..1.3e-7, Q6_K 1.5..1.6e-7 -> 1.1..1.2e-7, Q5_K 1.5..1.8e-7 -> 1.3..1.4e-7, Q3_K 1.5..1.6e-7 -> 0.9..1.0e-7)
bool gemv_wide_takes(const nh_device *d, const GemvArgs &a) {
    const int held = env_int("NEURA_HIP_GEMV_WIDE", 1);  // 0 never, 2 wherever it can
    if (held == 0 || a.rows < 2u || a.rows > 8u || a.rope || a.append_value || a.merge || a.digits_in || a.digits_out || a.pairs_out) return false;
    if (held != 2 && !few_narrow_rows_win(a.element, a.N, a.K, a.rows, a.swiglu, (uint32_t)d->compute_units)) return false;
    if ((uintptr_t)a.norm_w & 15u) return false;
    const uint32_t outputs = a.swiglu ? a.N / 2u : a.N;
    if (a.swiglu) return !a.residual && a.N % 2u == 0 && a.end[0] == outputs && a.W[1] && gemm_gates(d, a.element, outputs, a.K, whole_rows(a.rows), a.x, a.W[0], a.W[1]);
    return gemm_takes_whole(a.element, a.K, a.x, a.W[0]) && gemm_stacks(a.element, a.K, a.x, a.W[0], a.W[1], a.W[2], a.end[0], a.end[1]);
}

int32_t launch_gemv_wide(nh_device *d, const GemvArgs &a) {
    const uint32_t outputs = a.swiglu ? a.N / 2u : a.N;
    GemmArgs g{a.element, a.W[0], outputs, a.K, a.x, NH_F32, a.rows, a.y, a.residual, outputs};
    g.W_more[0] = a.W[1], g.W_more[1] = a.W[2], g.end[0] = a.end[0], g.end[1] = a.end[1];
    g.norm_w = a.norm_w, g.eps = a.eps, g.whole = true;
    if (a.swiglu) g.gated = true, g.W_more[1] = nullptr;
    return launch_gemm(d, g);
}

static int32_t launch_gemm_any(nh_device *d, const GemmArgs &a) {
    if (mfma_takes(a.element, a.K, a.X, a.W)) return launch_gemm_mfma(d, a);
    if (a.W_more[0] || a.W_more[1] || a.Y_more || a.packed || a.norm_w || a.gate || a.gated || a.whole)
        return fail(NH_E_ARGUMENT, "this wide product stacks no matrices, reuses no packed activations and packs rows as they lie (ask gemm_stacks first)");
    dim3 grid((a.N + BN - 1) / BN, (a.M + BM - 1) / BM), block(256);
    uint32_t row_bytes = (uint32_t)payload_bytes(a.element, a.K);
    const uint8_t *W = static_cast<const uint8_t *>(a.W);
    bool half = a.x_element == NH_F16;
#define NH_GEMM(E, H) hipLaunchKernelGGL((gemm_kernel<E, H>), grid, block, 0, d->stream, W, a.N, a.K, row_bytes, a.X, a.M, a.Y, a.residual, a.ldy)
    if (a.element == NH_Q8_0) {
        if (half) NH_GEMM(NH_Q8_0, true);
        else NH_GEMM(NH_Q8_0, false);
    } else if (a.element == NH_Q4_K) {
        if (half) NH_GEMM(NH_Q4_K, true);
        else NH_GEMM(NH_Q4_K, false);
    } else if (a.element == NH_Q6_K) {
        if (half) NH_GEMM(NH_Q6_K, true);
        else NH_GEMM(NH_Q6_K, false);
    } else if (a.element == NH_Q5_K) {
        if (half) NH_GEMM(NH_Q5_K, true);
        else NH_GEMM(NH_Q5_K, false);
    } else if (a.element == NH_Q3_K) {
        if (half) NH_GEMM(NH_Q3_K, true);
        else NH_GEMM(NH_Q3_K, false);
    } else {
        return fail(NH_E_ARGUMENT, "element %d carries no wide product", a.element);
    }
#undef NH_GEMM
    NH_HIP(hipGetLastError());
    return NH_OK;
}

int32_t launch_gemm(nh_device *d, const GemmArgs &a) {
    if (!a.M || !a.N) return NH_OK;
    // a narrow product's rows, or a step's products as nh_model_time_products counts them: one launch, its packing within
    const bool counted = a.whole || d->profile_wide;
    if (counted) profile_mark(d);
    if (const int32_t status = launch_gemm_any(d, a); status != NH_OK) return status;
    if (counted) profile_mark(d);
    if (counted && d->profile) d->profile_bytes += (uint64_t)a.N * (a.gated ? 2u : 1u) * payload_bytes(a.element, a.K);
    return NH_OK;
}

}  // namespace nh
