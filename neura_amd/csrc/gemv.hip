// Narrow products (one to eight activation rows, of Q4_K to sixteen; any count a few at a time) over raw GGUF blocks: y[r][n] = sum_k x[r][k] * W[n][k].
//
// Which Q4_K form a product reaches with no switch set (launch_gemv asks them in this order):
//
//   gemv_q4k_rows_kernel       3 to 16 activation rows, matrices that end on 16-row tiles, any K (deep rows in slices, which a fold adds up);
//                              q|k|v of three to sixteen planes with the rotation and the cache append in its epilogue (gemv_rows.hip)
//   gemv_q4k_tile16_kernel     1 row, any K of whole super-blocks, matrices that end on 16-row tiles: every product of a
//                              batch-1 decode step of the 0.5B .. 7B shapes; 2 rows where their digits fit LDS (ffn_down's 18944 columns
//                              included; the form above takes the rest) (gemv_tile16.hip)
//                              (with FIFTH the same for one row of Q5_K; gemv_q6k_tile16_kernel is its sibling for one row of Q6_K or Q3_K)
//   gemv_q4k_decode_kernel     1 row, K <= 4096, matrices that do NOT end on 16-row tiles or activations off a 16-byte
//                              boundary (odd vocabularies and widths: the small decoders of the tests); the vector form
//   gemv_q4k_kernel            the same refusals with K > 4096 or several rows: the LDS-tile vector form
//
// NEURA_HIP_TILE16=0, NEURA_HIP_MFMA=0 (the vector forms throughout) and NEURA_HIP_F16_TILES=0|2 push a product down (or up) this list so that the tests can hold the forms to each other on the same shapes.
//
// The vector form, Q4_K: a super-block is 144 B = a 16 B header (d, dmin, 12 scale bytes) + 128 B of nibbles.
// One lane owns one 64-element group of one super-block: it loads the header and its 32
// nibble bytes with three 128-bit loads, keeps its 64 activations in registers for the whole
// kernel and walks the output rows, so every weight byte is read from HBM exactly once and
// the activations never leave the register file.  A wave covers up to 16 super-blocks
// (4096 k); deeper rows are cut into slices whose partial sums a second kernel folds.
//
// Q8_0: 34 B blocks leave rows only 2-byte aligned, so a workgroup copies whole row slices
// into LDS with aligned 128-bit loads and each lane then reads its own block from LDS.
#include "blocks.hpp"
#include "common.hpp"
#include "gemv_shared.hpp"
#include "rows_rule.hpp"

#include <cstdlib>

namespace nh {

// skewed LDS index of activation i: 4 floats of padding per 64 keep 128-bit reads of
// neighbouring lanes on different banks
__device__ __forceinline__ uint32_t skew64(uint32_t i) { return i + (i >> 6) * 4; }
__device__ __forceinline__ uint32_t skew32(uint32_t i) { return i + (i >> 5) * 4; }

// 1 / sqrt(mean(x^2) + eps) of one activation row, to every thread.  Thread t adds columns t, t+256, ...
// as the reference's norm kernel does (crates/neura-kernel/src/task/norm.rs:69-83); the 256 partial
// sums are then joined inside each wave by shuffles and across waves through LDS with one barrier,
// not by the reference's eight-level tree (reduce.rs:21-38): a different order of the same fp32 adds.
__device__ float rms_scale(const float *__restrict__ x, uint32_t K, float eps, float *red) {
    float square = 0.0f;
    if (threadIdx.x < 256) {  // larger workgroups leave the sum to their first 256 threads
        for (uint32_t c = threadIdx.x; c < K; c += 256) {
            float value = x[c];
            square = __fadd_rn(square, __fmul_rn(value, value));
        }
    }
    square = wave_sum(square);
    if ((threadIdx.x & 63u) == 0 && threadIdx.x < 256) red[threadIdx.x >> 6] = square;
    __syncthreads();
    const float total = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();  // red is reused by the next row
    return rms_scale_of(total, K, eps);
}

// Stages x[k0 .. k0 + kn) of one activation row into LDS at dst[skew(i)], RMS-normalised over the whole row and
// weighed when norm_w is given.  With 256 threads and at most 32 values per thread every load goes out before the
// first value is used and the row is read once: a loop that handles each value as it arrives spends one memory
// round trip per value (6 us on a 3584-wide row).  Deeper slices take the looped form.
template <int PER, typename Skew>
__device__ __forceinline__ void stage_row_at_once(const float *__restrict__ x, uint32_t K, uint32_t k0, uint32_t kn, const float *__restrict__ norm_w,
                                                  float eps, float *dst, float *red, Skew skew) {
    const uint32_t tid = threadIdx.x;
    float held[PER], weight[PER];
    // every load is issued whatever its column (past the slice it reads the slice's last value, dropped below): loads
    // under a condition wait for one another
#pragma unroll
    for (int j = 0; j < PER; j++) held[j] = x[k0 + min(tid + 256u * j, kn - 1u)];
    if (norm_w) {
#pragma unroll
        for (int j = 0; j < PER; j++) weight[j] = norm_w[k0 + min(tid + 256u * j, kn - 1u)];
    }
#pragma unroll
    for (int j = 0; j < PER; j++)
        if (tid + 256u * j >= kn) held[j] = 0.0f;
    if (norm_w) {
        float square = 0.0f;  // thread t adds columns t, t + 256, ... in order (crates/neura-kernel/src/task/norm.rs:69-83)
#pragma unroll
        for (int j = 0; j < PER; j++) square = __fadd_rn(square, __fmul_rn(held[j], held[j]));
        square = wave_sum(square);
        if ((tid & 63u) == 0) red[tid >> 6] = square;
        __syncthreads();
        const float scale = rms_scale_of((red[0] + red[1]) + (red[2] + red[3]), K, eps);
        __syncthreads();  // red is reused by the next row
#pragma unroll
        for (int j = 0; j < PER; j++) held[j] = __fmul_rn(__fmul_rn(held[j], scale), weight[j]);
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const uint32_t c = tid + 256u * j;
        if (c < kn) dst[skew(c)] = held[j];
    }
}

// MOST: the values a thread holds at most (a kernel pays for its widest form in registers whether or not a launch takes it)
template <int MOST = 16, typename Skew>
__device__ __forceinline__ void stage_row(const float *__restrict__ x, uint32_t K, uint32_t k0, uint32_t kn, const float *__restrict__ norm_w,
                                          float eps, float *dst, float *red, Skew skew) {
    const uint32_t tid = threadIdx.x;
    const bool at_once = blockDim.x == 256 && kn > 0 && (!norm_w || (k0 == 0 && kn == K));
    if (at_once && kn <= 1024u) {  // no more loads than the slice needs, to the next power of two
        stage_row_at_once<4>(x, K, k0, kn, norm_w, eps, dst, red, skew);
    } else if (MOST >= 8 && at_once && kn <= 2048u) {
        stage_row_at_once<MOST >= 8 ? 8 : 4>(x, K, k0, kn, norm_w, eps, dst, red, skew);
    } else if (MOST >= 16 && at_once && kn <= 4096u) {
        stage_row_at_once<MOST >= 16 ? 16 : 4>(x, K, k0, kn, norm_w, eps, dst, red, skew);
    } else if (MOST >= 32 && at_once && kn <= 8192u) {
        stage_row_at_once<MOST >= 32 ? 32 : 4>(x, K, k0, kn, norm_w, eps, dst, red, skew);
    } else {
        float scale = 1.0f;
        if (norm_w) scale = rms_scale(x, K, eps, red);
        for (uint32_t i = tid; i < kn; i += blockDim.x) {
            float value = x[k0 + i];
            if (norm_w) value = __fmul_rn(__fmul_rn(value, scale), norm_w[k0 + i]);
            dst[skew(i)] = value;
        }
    }
}

// logical row i of a pass -> output row.  With swiglu, even i walk the gate rows and odd i the
// up rows so that one lane group ends up holding both halves of an output.
__device__ __forceinline__ uint32_t weight_row(uint32_t i, uint32_t N, int32_t swiglu) {
    return swiglu ? ((i & 1u) ? N / 2 + (i >> 1) : (i >> 1)) : i;
}

// first byte of output row n and the end of the matrix that holds it.  Written with selects
// over scalars: indexing the parameter arrays by a per-lane segment would turn into loads
// from the kernel argument block and serialise the weight loads behind them.
__device__ __forceinline__ const uint8_t *row_start(const GemvParams &p, uint32_t n, const uint8_t *&matrix_end) {
    const uint8_t *w0 = p.W[0], *w1 = p.W[1], *w2 = p.W[2];
    const uint32_t e0 = p.end[0], e1 = p.end[1], e2 = p.end[2];
    const bool first = n < e0, second = n < e1;
    const uint8_t *base = first ? w0 : (second ? w1 : w2);
    const uint32_t before = first ? 0u : (second ? e0 : e1);
    const uint32_t rows = first ? e0 : (second ? e1 - e0 : e2 - e1);
    matrix_end = base + (size_t)rows * p.row_bytes;
    return base + (size_t)(n - before) * p.row_bytes;
}

template <int R, int RB>
__device__ __forceinline__ void publish(const GemvParams &p, uint32_t first, uint32_t split, float (&acc)[R][RB]) {
    if (p.splits > 1) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            uint32_t i = first + r;
            if (i >= p.N) continue;
            uint32_t n = weight_row(i, p.N, p.swiglu);
#pragma unroll
            for (int b = 0; b < RB; b++) p.partial[((size_t)split * RB + b) * p.N + n] = acc[r][b];
        }
        return;
    }
    if (p.swiglu) {
#pragma unroll
        for (int r = 0; r + 1 < R; r += 2) {
            uint32_t i = first + r;
            if (i + 1 >= p.N) continue;
#pragma unroll
            for (int b = 0; b < RB; b++) p.y[(size_t)b * (p.N / 2) + (i >> 1)] = silu(acc[r][b]) * acc[r + 1][b];
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        uint32_t n = first + r;
        if (n >= p.N) continue;
#pragma unroll
        for (int b = 0; b < RB; b++) {
            float value = acc[r][b];
            if (p.residual) value = p.residual[(size_t)b * p.N + n] + value;
            p.y[(size_t)b * p.N + n] = value;
        }
    }
}

// ---------------------------------------------------------------------------- Q4_K -------


// Sum over the 32 low-nibble and the 32 high-nibble weights of 8 words against xl / xh.
// A nibble masked in place inside a 16-bit lane IS a half-precision subnormal: bits 0..3 read
// as code * 2^-24 and bits 4..7 as code * 2^-20, both exact.  The mixed-precision multiply-add
// (v_fma_mix_f32) widens the half operand on the fly, so a nibble costs one mask per pair and
// one multiply-add; the powers of two are folded into the block scales by the caller.
template <typename V4>
__device__ __forceinline__ void nibble_dots(const V4 &qa, const V4 &qb, const float (&xl)[32], const float (&xh)[32], float &low,
                                            float &high) {
    const uint32_t words[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
    float l = 0.0f, h = 0.0f;
#pragma unroll
    for (int w = 0; w < 8; w++) {
        const uint32_t even = words[w], odd = words[w] >> 8;  // bytes (0, 2) and bytes (1, 3) in the 16-bit lanes
        const half2_t l02 = __builtin_bit_cast(half2_t, even & 0x000f000fu);
        const half2_t h02 = __builtin_bit_cast(half2_t, even & 0x00f000f0u);
        const half2_t l13 = __builtin_bit_cast(half2_t, odd & 0x000f000fu);
        const half2_t h13 = __builtin_bit_cast(half2_t, odd & 0x00f000f0u);
        l = fmaf((float)l02.x, xl[4 * w + 0], l);
        l = fmaf((float)l13.x, xl[4 * w + 1], l);
        l = fmaf((float)l02.y, xl[4 * w + 2], l);
        l = fmaf((float)l13.y, xl[4 * w + 3], l);
        h = fmaf((float)h02.x, xh[4 * w + 0], h);
        h = fmaf((float)h13.x, xh[4 * w + 1], h);
        h = fmaf((float)h02.y, xh[4 * w + 2], h);
        h = fmaf((float)h13.y, xh[4 * w + 3], h);
    }
    low = l;   // scaled by 2^-24: the caller folds 2^24 into xl or the block scale
    high = h;  // scaled by 2^-20
}

// the two (scale, min) pairs of group g (sub-blocks 2g and 2g+1) from a block header
__device__ __forceinline__ void group_scales(const uint4 &hdr, uint32_t g, float &d0, float &d1, float &m0, float &m1) {
    float d = half_to_float((uint16_t)(hdr.x & 0xffffu));
    float dmin = half_to_float((uint16_t)(hdr.x >> 16));
    uint32_t shift = 16u * (g & 1u);
    uint32_t ya = (hdr.y >> shift) & 0xffffu, za = (hdr.z >> shift) & 0xffffu, wa = (hdr.w >> shift) & 0xffffu;
    uint32_t sc0, sc1, mn0, mn1;
    if (g < 2) {
        sc0 = ya & 63u;
        sc1 = (ya >> 8) & 63u;
        mn0 = za & 63u;
        mn1 = (za >> 8) & 63u;
    } else {
        sc0 = (wa & 0x0fu) | (((ya >> 6) & 3u) << 4);
        sc1 = ((wa >> 8) & 0x0fu) | (((ya >> 14) & 3u) << 4);
        mn0 = ((wa >> 4) & 0x0fu) | (((za >> 6) & 3u) << 4);
        mn1 = ((wa >> 12) & 0x0fu) | (((za >> 14) & 3u) << 4);
    }
    d0 = d * (float)sc0;
    d1 = d * (float)sc1;
    m0 = dmin * (float)mn0;
    m1 = dmin * (float)mn1;
}

// Sums R per-lane partials over the G lanes of a row group.  The first log2(R) steps fold two
// rows into one register (each lane keeps the row its own index selects), so R rows cost
// R - 1 + log2(G / R) exchanges instead of R log2(G); steps inside a row of 16 lanes are DPP
// adds, only the steps across 16 and 32 lanes go through the LDS crossbar.  On return lane u
// (u < R, u = lane % G) of every group holds the total of row u.
template <int R, int G>
__device__ __forceinline__ float fold_rows(float (&acc)[R], uint32_t lane) {
    static_assert(R == 2 || R == 4, "rows per pass");
    static_assert(G == 16 || G == 32 || G == 64, "lanes per row group");
    float v;
    const bool odd = lane & 1u;
    if (R == 4) {
        const bool upper = lane & 2u;
        float keep01 = odd ? acc[1] : acc[0], send01 = odd ? acc[0] : acc[1];
        float keep23 = odd ? acc[3] : acc[2], send23 = odd ? acc[2] : acc[3];
        float v01 = keep01 + dpp<DPP_QUAD_XOR1>(send01);
        float v23 = keep23 + dpp<DPP_QUAD_XOR1>(send23);
        float keep = upper ? v23 : v01, send = upper ? v01 : v23;
        v = keep + dpp<DPP_QUAD_XOR2>(send);
    } else {
        float keep = odd ? acc[1] : acc[0], send = odd ? acc[0] : acc[1];
        v = keep + dpp<DPP_QUAD_XOR1>(send);
        v += dpp<DPP_QUAD_XOR2>(v);
    }
    v += dpp<DPP_ROW_ROR4>(v);  // rotations inside a row of 16 lanes keep lane % 4
    v += dpp<DPP_ROW_ROR8>(v);
    if (G >= 32) v += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));  // lane ^ 16
    if (G >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

// The epilogue of a q|k|v product that folds the rotation in: lane u < R of a lane group holds logical row i = first + u, and
// logical rows 2t, 2t + 1 are channels c and c + width/2 of one head (crates/neura-kernel/src/task/rope.rs:95-122).  The
// projection's bias, if it has one, comes before the rotation; q rows go to y, k rows rotated and v rows as they are to the
// caches as halves, at the cursor (at cursor mod span in a ring).  Every lane of the wave calls it.
template <int R>
__device__ __forceinline__ void rotate_and_store(const GemvParams &p, float total, uint32_t i, uint32_t u) {
    const uint32_t half = p.rope_width >> 1, pair = min(i, p.N - 1u) >> 1, c = pair % half;
    const uint32_t n = (pair / half) * p.rope_width + c + (i & 1u) * half;
    if (u < R && i < p.N) {
        const float *b0 = p.bias[0], *b1 = p.bias[1], *b2 = p.bias[2];
        const uint32_t e0 = p.end[0], e1 = p.end[1];
        const float *bias = n < e0 ? b0 : (n < e1 ? b1 : b2);
        const uint32_t before = n < e0 ? 0u : (n < e1 ? e0 : e1);
        if (bias) total += bias[n - before];
    }
    const float other = dpp<DPP_QUAD_XOR1>(total);
    if (u < R && i < p.N) {
        const uint32_t position = p.rope_cursor[0];
        float value = total;
        if (n < p.rope_k_rows) {
            // cos and sin of f32(position) * pow(base, -2c/width), tabulated once per model by the rotation's own kernel
            const float cosine = p.rope_cosines[(size_t)min(position, p.rope_positions - 1u) * half + c];
            const float sine = p.rope_sines[(size_t)min(position, p.rope_positions - 1u) * half + c];
            value = (i & 1u) ? total * cosine + other * sine : total * cosine - other * sine;
        }
        if (n < p.rope_q_rows) {
            p.y[n] = value;
        } else if (position >= p.rope_positions || (!p.rope_ring && position >= p.rope_capacity)) {
            atomicMax(p.refusal, (uint32_t)REFUSAL_ORIGIN);
        } else {
            const bool key = n < p.rope_k_rows;
            const uint32_t within = n - (key ? p.rope_q_rows : p.rope_k_rows);  // head * width + channel
            const uint32_t head = within / p.rope_width, channel = within % p.rope_width;
            uint16_t *cache = key ? p.rope_k : p.rope_v;
            const uint32_t slot = p.rope_ring ? position % p.rope_ring : position;  // a ring seats position p at p mod its span
            state_store(cache, p.rope_element, ((uint64_t)head * p.rope_capacity + slot) * p.rope_width + channel, value);
        }
    }
}

// One pass of the decode kernel over R rows: the raw blocks a lane owns.
template <int R>
struct DecodeTile {
    u32x4 hdr[R], qa[R], qb[R];
};

// Decode path (one activation row).  G = lanes per output row (64: one row group per wave
// pass, the hot case; 32 / 16: short rows, several row groups side by side in a wave).
//
// A lane owns one 64-element group of one super-block for the whole kernel and keeps its 64
// activations in registers.  Every integer field is consumed as a half-precision subnormal by
// mixed-precision multiply-adds (nibbles: * 2^-24 / 2^-20, undone by scaling the activations
// once; scales: * 2^-24, undone once per pass), so a weight costs 1.6 vector instructions.
template <int R, int G, bool PIPE, int NW, bool ROPE = false>
__global__ __launch_bounds__(NW * 64) void gemv_q4k_decode_kernel(GemvParams p) {
    extern __shared__ float xs[];  // skew64(slice)
    __shared__ float red[256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t split = blockIdx.y;
    const uint32_t blk0 = split * p.blocks_per_split;
    const uint32_t nb = min(p.blocks_per_split, p.nblk - blk0);
    const uint32_t k0 = blk0 * 256u, kn = nb * 256u;

    constexpr uint32_t RS = 64u / G;
    constexpr uint32_t rows_per_pass = R * RS;
    const uint32_t u = lane & (G - 1u), rs = lane / G;
    const bool active = u < nb * 4u;
    const uint32_t unit = active ? u : 0u;  // an idle lane re-reads unit 0 against zero activations
    const uint32_t g = unit & 3u;
    const uint32_t lane_offset = (blk0 + (unit >> 2)) * 144u + g * 32u;
    const ScaleLane lane_scales = scale_lane(g);

    auto load = [&](DecodeTile<R> &t, uint32_t rg) {
        const uint32_t first = rg * rows_per_pass + rs * R;  // first logical row of this lane group (a multiple of R)
        // R rows of one matrix: rows never straddle a matrix (every end is a multiple of R)
        const uint8_t *base[R];
        if (p.swiglu) {
            const uint32_t pair = min(first, p.N - R) >> 1;  // logical rows 2q, 2q+1 = gate row q, up row q
#pragma unroll
            for (int r = 0; r < R; r++) base[r] = ((r & 1) ? p.W[1] : p.W[0]) + (size_t)(pair + (r >> 1)) * p.row_bytes;
        } else {
            // with the rotation folded in, logical rows 2t, 2t+1 are channels t and t + width/2 of one head
            const uint32_t logical = min(first, p.N - R);
            const uint32_t half = p.rope_width >> 1, pair = logical >> 1;
            const uint32_t n = ROPE ? (pair / half) * p.rope_width + pair % half : logical;
            const uint32_t hop = ROPE ? half : 1u;
            const bool in0 = n < p.end[0], in1 = n < p.end[1];
            const uint8_t *matrix = in0 ? p.W[0] : (in1 ? p.W[1] : p.W[2]);
            const uint32_t before = in0 ? 0u : (in1 ? p.end[0] : p.end[1]);
#pragma unroll
            for (int r = 0; r < R; r++) base[r] = matrix + (size_t)(n - before + r * hop) * p.row_bytes;
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            typedef const __attribute__((address_space(1))) u32x4 *global_uint4;  // the arena is global memory
            const uint8_t *at = base[r] + lane_offset;
            t.hdr[r] = *(global_uint4)(uintptr_t)(at - g * 32u);
            t.qa[r] = *(global_uint4)(uintptr_t)(at + 16u);
            t.qb[r] = *(global_uint4)(uintptr_t)(at + 32u);
        }
    };

    const uint32_t stride = gridDim.x * NW;
    uint32_t rg = blockIdx.x * NW + wave;
    DecodeTile<R> ta, tb;
    if (rg < p.row_groups) load(ta, rg);  // in flight while the activations are staged

    stage_row(p.x, p.K, k0, kn, p.norm_w, p.eps, xs, red, [](uint32_t i) { return skew64(i); });
    __syncthreads();

    float xl[32], xh[32];
    float xsl = 0.0f, xsh = 0.0f;  // plain sums of this lane's activations (for the block minimums)
    {
        const float4 *src = reinterpret_cast<const float4 *>(xs + skew64(unit * 64u));
        const float keep = active ? 1.0f : 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // sum and scale each chunk as it arrives: raw and scaled copies never coexist
            float4 a = src[j], c = src[8 + j];
            xsl += (a.x + a.y) + (a.z + a.w);
            xsh += (c.x + c.y) + (c.z + c.w);
            const float sl = keep * 16777216.0f, sh = keep * 1048576.0f;  // nibbles arrive * 2^-24 / * 2^-20
            xl[4 * j] = a.x * sl, xl[4 * j + 1] = a.y * sl, xl[4 * j + 2] = a.z * sl, xl[4 * j + 3] = a.w * sl;
            xh[4 * j] = c.x * sh, xh[4 * j + 1] = c.y * sh, xh[4 * j + 2] = c.z * sh, xh[4 * j + 3] = c.w * sh;
        }
        xsl *= keep, xsh *= keep;
    }

    auto compute = [&](const DecodeTile<R> &t, uint32_t rg) {
        const uint32_t first = rg * rows_per_pass + rs * R;
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            float low, high;
            nibble_dots(t.qa[r], t.qb[r], xl, xh, low, high);
            half2_t sc, mn;
            scale_pairs(t.hdr[r], lane_scales, sc, mn);
            const half2_t dd = __builtin_bit_cast(half2_t, t.hdr[r].x);  // (d, dmin)
            const float weighed = fmaf((float)sc.y, high, (float)sc.x * low);
            const float floor_ = fmaf((float)mn.y, xsh, (float)mn.x * xsl);
            acc[r] = fmaf((float)dd.x, weighed, -((float)dd.y * floor_));
        }
        float total = fold_rows<R, G>(acc, lane) * 16777216.0f;  // the scales arrived * 2^-24
        const uint32_t i = first + u;                             // lane u < R holds row first + u
        if (p.splits > 1) {
            if (u < R && i < p.N) p.partial[(size_t)split * p.N + weight_row(i, p.N, p.swiglu)] = total;
        } else if (p.swiglu) {
            float up = dpp<DPP_QUAD_XOR1>(total);
            if (u < R && !(u & 1u) && i + 1 < p.N) p.y[i >> 1] = silu(total) * up;
        } else if (ROPE) {
            rotate_and_store<R>(p, total, i, u);
        } else if (u < R && i < p.N) {
            p.y[i] = p.residual ? p.residual[i] + total : total;
        }
    };

    if (PIPE) {
        while (rg < p.row_groups) {
            uint32_t next = rg + stride;
            if (next < p.row_groups) load(tb, next);
            compute(ta, rg);
            rg = next;
            if (rg >= p.row_groups) break;
            next = rg + stride;
            if (next < p.row_groups) load(ta, next);
            compute(tb, rg);
            rg = next;
        }
    } else {
        while (rg < p.row_groups) {
            compute(ta, rg);
            rg += stride;
            __builtin_amdgcn_sched_barrier(0);  // the next loads reuse this tile's registers: keep them behind the arithmetic
            if (rg < p.row_groups) load(ta, rg);
        }
    }
}

// General narrow product: RB activation rows (2 or 4) staged in LDS and re-read per row group.
template <int R, int RB>
__global__ __launch_bounds__(256) void gemv_q4k_kernel(GemvParams p) {
    fetch_parameters(p);
    extern __shared__ float xs[];  // [RB][skew64(slice)]
    __shared__ float red[256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t split = blockIdx.y;
    const uint32_t blk0 = split * p.blocks_per_split;
    const uint32_t nb = min(p.blocks_per_split, p.nblk - blk0);
    const uint32_t k0 = blk0 * 256u, kn = nb * 256u;
    const uint32_t xstride = skew64(p.blocks_per_split * 256u);

#pragma unroll
    for (int b = 0; b < RB; b++)
        stage_row(p.x + (size_t)b * p.K, p.K, k0, kn, p.norm_w, p.eps, xs + b * xstride, red, [](uint32_t i) { return skew64(i); });
    __syncthreads();

    const uint32_t G = p.group;  // lanes per output row
    const uint32_t u = lane & (G - 1u), rs = lane / G, RS = 64u / G;
    const bool active = u < nb * 4u;
    const uint32_t blk = active ? (u >> 2) : 0u, g = u & 3u;
    float xl[32], xh[32];

    const uint32_t rows_per_pass = R * RS;
    for (uint32_t rg = blockIdx.x * 4u + wave; rg < p.row_groups; rg += gridDim.x * 4u) {
        const uint32_t first = rg * rows_per_pass + rs * R;  // first logical row of this lane group
        uint4 hdr[R], qa[R], qb[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            uint32_t i = first + r;
            uint32_t n = weight_row(i < p.N ? i : 0u, p.N, p.swiglu);
            const uint8_t *matrix_end;
            const uint8_t *base = row_start(p, n, matrix_end) + (size_t)(blk0 + blk) * 144u;
            hdr[r] = *reinterpret_cast<const uint4 *>(base);
            qa[r] = *reinterpret_cast<const uint4 *>(base + 16u + g * 32u);
            qb[r] = *reinterpret_cast<const uint4 *>(base + 32u + g * 32u);
        }
        float acc[R][RB];
#pragma unroll
        for (int b = 0; b < RB; b++) {
            const float4 *src = reinterpret_cast<const float4 *>(xs + b * xstride + skew64((blk * 4u + g) * 64u));
            float xsl = 0.0f, xsh = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float4 a = active ? src[j] : make_float4(0.f, 0.f, 0.f, 0.f);
                float4 c = active ? src[8 + j] : make_float4(0.f, 0.f, 0.f, 0.f);
                xl[4 * j] = a.x, xl[4 * j + 1] = a.y, xl[4 * j + 2] = a.z, xl[4 * j + 3] = a.w;
                xh[4 * j] = c.x, xh[4 * j + 1] = c.y, xh[4 * j + 2] = c.z, xh[4 * j + 3] = c.w;
            }
#pragma unroll
            for (int j = 0; j < 32; j++) xsl += xl[j], xsh += xh[j];
#pragma unroll
            for (int r = 0; r < R; r++) {
                float d0, d1, m0, m1, low, high;
                group_scales(hdr[r], g, d0, d1, m0, m1);
                nibble_dots(qa[r], qb[r], xl, xh, low, high);
                acc[r][b] = (d0 * (low * 16777216.0f) + d1 * (high * 1048576.0f)) - (m0 * xsl + m1 * xsh);
            }
        }
        // sum over the G lanes of the group
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int b = 0; b < RB; b++) {
                float v = acc[r][b];
                for (uint32_t offset = G >> 1; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, 64);
                acc[r][b] = v;
            }
        if (u == 0) publish<R, RB>(p, first, split, acc);
    }
}

// ---------------------------------------------------------------------------- Q8_0 -------

template <int R, int RB>
__global__ __launch_bounds__(256) void gemv_q8_0_kernel(GemvParams p) {
    fetch_parameters(p);
    extern __shared__ float shared[];  // xs [RB][skew32(slice)] then the staged weight tile
    __shared__ float red[256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t split = blockIdx.y;
    const uint32_t blk0 = split * p.blocks_per_split;
    const uint32_t nb = min(p.blocks_per_split, p.nblk - blk0);
    const uint32_t k0 = blk0 * 32u, kn = nb * 32u;
    const uint32_t xstride = skew32(p.blocks_per_split * 32u);
    float *xs = shared;
    uint8_t *tile = reinterpret_cast<uint8_t *>(shared + RB * xstride);  // 16-byte aligned: xstride is a multiple of 4
    const uint32_t lrow = p.chunks_per_row * 16u;

#pragma unroll
    for (int b = 0; b < RB; b++)
        stage_row(p.x + (size_t)b * p.K, p.K, k0, kn, p.norm_w, p.eps, xs + b * xstride, red, [](uint32_t i) { return skew32(i); });
    __syncthreads();

    const uint32_t G = p.group;
    const uint32_t u = lane & (G - 1u), rs = lane / G, RS = 64u / G;
    const bool active = u < nb;

    float xr[32];
    float xsum = 0.0f;
    if (RB == 1) {
        const float4 *src = reinterpret_cast<const float4 *>(xs + skew32((active ? u : 0u) * 32u));
#pragma unroll
        for (int j = 0; j < 8; j++) {
            float4 a = active ? src[j] : make_float4(0.f, 0.f, 0.f, 0.f);
            xr[4 * j] = a.x, xr[4 * j + 1] = a.y, xr[4 * j + 2] = a.z, xr[4 * j + 3] = a.w;
        }
#pragma unroll
        for (int j = 0; j < 32; j++) xsum += xr[j];
    }

    const uint32_t rows_per_wave = R * RS, rows_per_tile = rows_per_wave * 4u;
    const uint32_t slice_bytes = nb * 34u;
    const uint32_t tiles = (p.row_groups + 3u) / 4u;  // row_groups counts wave passes
    for (uint32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        const uint32_t tile_first = t * rows_per_tile;
        __syncthreads();  // the previous tile is no longer read
        for (uint32_t c = tid; c < rows_per_tile * p.chunks_per_row; c += 256) {
            uint32_t local = c / p.chunks_per_row, chunk = c % p.chunks_per_row;
            uint32_t i = tile_first + local;
            if (i >= p.N) continue;
            uint32_t n = weight_row(i, p.N, p.swiglu);
            const uint8_t *w_end;
            const uint8_t *start = row_start(p, n, w_end) + (size_t)blk0 * 34u;
            const uint8_t *aligned = start - ((uintptr_t)start & 15u);
            uint32_t lead = (uint32_t)((uintptr_t)start & 15u);
            if (chunk * 16u >= lead + slice_bytes) continue;
            const uint8_t *src = aligned + chunk * 16u;
            uint4 held;
            if (src + 16 <= w_end) {
                held = *reinterpret_cast<const uint4 *>(src);
            } else {  // the last bytes of the tensor: never read past its end
                uint8_t bytes[16];
#pragma unroll
                for (int j = 0; j < 16; j++) bytes[j] = (src + j < w_end) ? src[j] : (uint8_t)0;
                held = *reinterpret_cast<uint4 *>(bytes);
            }
            *reinterpret_cast<uint4 *>(tile + local * lrow + chunk * 16u) = held;
        }
        __syncthreads();

        const uint32_t local_first = wave * rows_per_wave + rs * R;
        const uint32_t first = tile_first + local_first;
        float acc[R][RB];
        uint32_t quants[R][8];
        float scales[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            uint32_t i = first + r;
            uint32_t n = weight_row(i < p.N ? i : 0u, p.N, p.swiglu);
            const uint8_t *matrix_end;
            uint32_t lead = (uint32_t)((uintptr_t)(row_start(p, n, matrix_end) + (size_t)blk0 * 34u) & 15u);
            uint32_t at = (local_first + r) * lrow + lead + (active ? u : 0u) * 34u;  // byte offset of the block in the tile
            bool held = active && i < p.N;
            scales[r] = held ? half_to_float(*reinterpret_cast<const uint16_t *>(tile + at)) : 0.0f;
            uint32_t payload = at + 2u;
            const uint32_t *words = reinterpret_cast<const uint32_t *>(tile + (payload & ~3u));
            uint32_t shift = (payload & 3u) * 8u;  // 0 or 16
            uint32_t raw[9];
#pragma unroll
            for (int j = 0; j < 9; j++) raw[j] = held ? words[j] : 0u;
#pragma unroll
            for (int j = 0; j < 8; j++) quants[r][j] = __funnelshift_r(raw[j], raw[j + 1], shift) ^ 0x80808080u;  // q + 128
        }
#pragma unroll
        for (int b = 0; b < RB; b++) {
            if (RB > 1) {
                const float4 *src = reinterpret_cast<const float4 *>(xs + b * xstride + skew32((active ? u : 0u) * 32u));
                xsum = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    float4 a = active ? src[j] : make_float4(0.f, 0.f, 0.f, 0.f);
                    xr[4 * j] = a.x, xr[4 * j + 1] = a.y, xr[4 * j + 2] = a.z, xr[4 * j + 3] = a.w;
                }
#pragma unroll
                for (int j = 0; j < 32; j++) xsum += xr[j];
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                float total = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    uint32_t w = quants[r][j];
                    total = fmaf(xr[4 * j + 0], (float)(w & 0xffu), total);
                    total = fmaf(xr[4 * j + 1], (float)((w >> 8) & 0xffu), total);
                    total = fmaf(xr[4 * j + 2], (float)((w >> 16) & 0xffu), total);
                    total = fmaf(xr[4 * j + 3], (float)(w >> 24), total);
                }
                acc[r][b] = scales[r] * (total - 128.0f * xsum);
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int b = 0; b < RB; b++) {
                float v = acc[r][b];
                for (uint32_t offset = G >> 1; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, 64);
                acc[r][b] = v;
            }
        if (u == 0) publish<R, RB>(p, first, split, acc);
    }
}

// The activation row of the product behind a decode attention, merged from the sums the attention left a section of the keys
// each (SectionSums; crates/neura-kernel/src/task/attention.rs:619-671 is the merge): element (head, channel) is the sections'
// channel sums weighed by e^(section's largest score - the largest of all) over the masses weighed the same way.  Every load
// a thread needs -- the statistics of two (head, section) pairs, sixteen channel sums of each of its four elements -- is asked
// for before the first is used (sections past the last read the last again and are dropped).  The statistics cross in LDS:
// the thread of a pair turns its section's largest score into the section's weight, the thread of an element then reads
// sixteen weights and masses.  `width` is a power of two (the decode attention's 64 or 128).
template <typename Skew>
__device__ __forceinline__ void stage_merged(const float *__restrict__ partial, uint32_t sections, uint32_t G, uint32_t width, uint32_t K, float *xs, Skew skew) {
    constexpr uint32_t MOST = MERGED_SECTIONS_MOST, HEADS_MOST = 32;
    __shared__ __attribute__((aligned(16))) float tops[HEADS_MOST * MOST], masses[HEADS_MOST * MOST], weights[HEADS_MOST * MOST];
    const uint32_t tid = threadIdx.x, shift = 31u - __builtin_clz(width), heads = K >> shift, hop = G * (width + 2u);
    const uint32_t by_groups = 65536u / G + 1u;  // x / G = x * by_groups >> 16 for the few heads here
    auto sums_of = [&](uint32_t head) {
        const uint32_t unit = head * by_groups >> 16;
        return partial + ((uint64_t)unit * sections * G + (head - unit * G)) * (width + 2u);
    };
    // seat tid + 256 j of the statistics: head seat / MOST, section seat % MOST; a seat past the heads or the sections holds
    // no score and no mass (its loads read the last head's, the last section's, and are dropped)
    float top[2], mass[2];
    bool seated[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t seat = tid + 256u * j, head = seat / MOST, section = seat % MOST;
        seated[j] = head < heads && section < sections;
        const float *stats = sums_of(min(head, heads - 1u)) + min(section, sections - 1u) * hop + width;
        top[j] = stats[0], mass[j] = stats[1];
    }
    for (uint32_t base = 0; base < K; base += 1024u) {
        float values[4][MOST];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t i = min(base + tid + 256u * e, K - 1u);
            const float *column = sums_of(i >> shift) + (i & (width - 1u));
#pragma unroll
            for (uint32_t s = 0; s < MOST; s++) values[e][s] = column[min(s, sections - 1u) * hop];
        }
        if (base == 0) {
#pragma unroll
            for (int j = 0; j < 2; j++) tops[tid + 256u * j] = seated[j] ? top[j] : -INFINITY, masses[tid + 256u * j] = seated[j] ? mass[j] : 0.0f;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float4 *row = reinterpret_cast<const float4 *>(tops + ((tid + 256u * j) & ~(MOST - 1u)));
                float largest = -INFINITY;
#pragma unroll
                for (uint32_t q = 0; q < MOST / 4u; q++) largest = fmaxf(fmaxf(largest, fmaxf(row[q].x, row[q].y)), fmaxf(row[q].z, row[q].w));
                weights[tid + 256u * j] = !seated[j] || top[j] == -INFINITY ? 0.0f : softmax_exp(top[j] - largest);
            }
            __syncthreads();
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t i = base + tid + 256u * e;
            if (i >= K) continue;
            const float4 *head_weights = reinterpret_cast<const float4 *>(weights + (i >> shift) * MOST);
            const float4 *head_masses = reinterpret_cast<const float4 *>(masses + (i >> shift) * MOST);
            float total = 0.0f, sum = 0.0f;
#pragma unroll
            for (uint32_t q = 0; q < MOST / 4u; q++) {
                const float4 w = head_weights[q], m = head_masses[q];
                total = fmaf(m.x, w.x, total), total = fmaf(m.y, w.y, total), total = fmaf(m.z, w.z, total), total = fmaf(m.w, w.w, total);
                sum = fmaf(values[e][4 * q], w.x, sum), sum = fmaf(values[e][4 * q + 1], w.y, sum);
                sum = fmaf(values[e][4 * q + 2], w.z, sum), sum = fmaf(values[e][4 * q + 3], w.w, sum);
            }
            xs[skew(i)] = total > 0.0f ? sum * (1.0f / total) : 0.0f;
        }
    }
}

// Q8_0, one activation row, rows of at most 64 blocks (K <= 2048): the shape of the Q4_K decode kernel.  A lane owns one
// block column for the whole kernel and keeps its 32 activations in registers; the 34 bytes of a block sit on a 2-byte
// boundary, so a lane reads the nine words that cover it from the 4-byte boundary below it (the reference's own reading,
// crates/neura-kernel/src/dot.rs:197-264) and realigns by 16 bits where the block starts on a half word.  No LDS tile and no
// barrier between the rows: the first pass's words are on their way while the activations are staged.
typedef uint32_t u32x4_loose __attribute__((ext_vector_type(4), aligned(4)));

template <int R>
struct Q8Tile {
    u32x4 a[R], b[R];
    uint32_t c[R];
    uint32_t odd[R];  // 2 where the row's block starts on a half word, else 0
};

// DEEP (rows of 65 to 256 blocks, K <= 8192): the four waves of a workgroup walk the same rows, wave w the blocks 64 w ..
// 64 w + 63, and meet in LDS once a pass.
// The leading arguments are what the first weight loads and the activations' need: plain words the hardware hands to a wave in
// scalar registers as it starts (Q8_LEAD packs them: the rotation's width rides above the blocks a row, the SwiGLU flag above
// N); they take the place of the same members of the parameter block, whose other members are loaded as they come to use.
#define Q8_LEAD(p) (p).W[0], (p).W[1], (p).W[2], (p).x, (p).row_bytes, (p).nblk | ((p).rope_width << 16), (p).row_groups, (p).N | ((p).swiglu ? 0x80000000u : 0u), (p).end[0], (p).end[1], (p)
// MERGE: the activation row is merged from a decode attention's section sums (x points at them) as it is staged.
template <int R, int G, bool DEEP = false, bool ROPE = false, bool MERGE = false>
__global__ __launch_bounds__(256) void gemv_q8_0_decode_kernel(const uint8_t *lead_w0, const uint8_t *lead_w1, const uint8_t *lead_w2, const float *lead_x,
                                                               uint32_t lead_row_bytes, uint32_t lead_nblk_width, uint32_t lead_row_groups, uint32_t lead_n_swiglu,
                                                               uint32_t lead_end0, uint32_t lead_end1, GemvParams rest) {
    GemvParams p = rest;
    p.W[0] = lead_w0, p.W[1] = lead_w1, p.W[2] = lead_w2, p.x = lead_x, p.row_bytes = lead_row_bytes, p.row_groups = lead_row_groups;
    p.nblk = lead_nblk_width & 0xffffu, p.rope_width = lead_nblk_width >> 16, p.K = 32u * (lead_nblk_width & 0xffffu);
    p.N = lead_n_swiglu & 0x7fffffffu, p.swiglu = (int32_t)(lead_n_swiglu >> 31), p.end[0] = lead_end0, p.end[1] = lead_end1;
    static_assert(!DEEP || G == 64, "a deep row fills every wave");
    static_assert(!ROPE || (R == 2 && !DEEP), "the rotation pairs the two rows of a pass");
    extern __shared__ float xs[];  // skew32(K)
    __shared__ float red[256];
    __shared__ float part[2][4][R];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr uint32_t RS = 64u / G, rows_per_pass = R * RS;
    const uint32_t u = lane & (G - 1u), rs = lane / G;
    const uint32_t block = DEEP ? 64u * wave + u : u;
    const bool active = block < p.nblk;
    const uint32_t unit = active ? block : 0u;  // an idle lane re-reads block 0 against zero activations

    auto load = [&](Q8Tile<R> &t, uint32_t rg) {
        const uint32_t first = rg * rows_per_pass + rs * R;  // first logical row of this lane group (a multiple of R)
        const uint8_t *base[R];
        if (p.swiglu) {
            const uint32_t pair = min(first, p.N - R) >> 1;  // logical rows 2q, 2q+1 = gate row q, up row q
#pragma unroll
            for (int r = 0; r < R; r++) base[r] = ((r & 1) ? p.W[1] : p.W[0]) + (size_t)(pair + (r >> 1)) * p.row_bytes;
        } else {
            // R rows of one matrix: every matrix end is a multiple of R.  With the rotation folded in, logical rows 2t, 2t+1
            // are channels t and t + width/2 of one head
            const uint32_t logical = min(first, p.N - R);
            const uint32_t half = p.rope_width >> 1, pair = logical >> 1;
            const uint32_t n = ROPE ? (pair / half) * p.rope_width + pair % half : logical;
            const uint32_t hop = ROPE ? half : 1u;
            const bool in0 = n < p.end[0], in1 = n < p.end[1];
            const uint8_t *matrix = in0 ? p.W[0] : (in1 ? p.W[1] : p.W[2]);
            const uint32_t before = in0 ? 0u : (in1 ? p.end[0] : p.end[1]);
#pragma unroll
            for (int r = 0; r < R; r++) base[r] = matrix + (size_t)(n - before + r * hop) * p.row_bytes;
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uintptr_t at = (uintptr_t)(base[r] + unit * 34u);
            const uintptr_t low = at & ~(uintptr_t)3;
            t.odd[r] = (uint32_t)(at & 2u);
            t.a[r] = *(const __attribute__((address_space(1))) u32x4_loose *)low;
            t.b[r] = *(const __attribute__((address_space(1))) u32x4_loose *)(low + 16u);
            // a block on a word boundary ends two bytes into the ninth word: those two only are read (the last block of a
            // tensor ends where its allocation may)
            if (at & 2u) t.c[r] = *(const __attribute__((address_space(1))) uint32_t *)(low + 32u);
            else t.c[r] = *(const __attribute__((address_space(1))) uint16_t *)(low + 32u);
        }
    };

    const uint32_t stride = DEEP ? gridDim.x : gridDim.x * 4u;
    uint32_t rg = DEEP ? blockIdx.x : blockIdx.x * 4u + wave;
    uint32_t parity = 0;
    Q8Tile<R> held;
    if (rg < p.row_groups) load(held, rg);  // in flight while the activations are staged

    if constexpr (MERGE) stage_merged(p.x, p.merge_sections, p.merge_groups, p.merge_width, p.K, xs, [](uint32_t i) { return skew32(i); });
    else stage_row<DEEP ? 32 : 8>(p.x, p.K, 0u, p.K, p.norm_w, p.eps, xs, red, [](uint32_t i) { return skew32(i); });  // rows of 256 blocks, or of 64
    __syncthreads();

    float xr[32];
    float xsum = 0.0f;
    {
        const float4 *src = reinterpret_cast<const float4 *>(xs + skew32(unit * 32u));
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float4 a = active ? src[j] : make_float4(0.f, 0.f, 0.f, 0.f);
            xr[4 * j] = a.x, xr[4 * j + 1] = a.y, xr[4 * j + 2] = a.z, xr[4 * j + 3] = a.w;
        }
#pragma unroll
        for (int j = 0; j < 32; j++) xsum += xr[j];
    }

    while (rg < p.row_groups) {
        const uint32_t first = rg * rows_per_pass + rs * R;
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t words[9] = {held.a[r].x, held.a[r].y, held.a[r].z, held.a[r].w, held.b[r].x, held.b[r].y, held.b[r].z, held.b[r].w, held.c[r]};
            const bool odd = held.odd[r] != 0u;
            // the scale is the half at the block's first two bytes, the 32 codes follow it
            const float scale = half_to_float((uint16_t)(odd ? words[0] >> 16 : words[0] & 0xffffu));
            float total = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t w = (odd ? words[j + 1] : __funnelshift_r(words[j], words[j + 1], 16)) ^ 0x80808080u;  // q + 128
                total = fmaf(xr[4 * j + 0], (float)(w & 0xffu), total);
                total = fmaf(xr[4 * j + 1], (float)((w >> 8) & 0xffu), total);
                total = fmaf(xr[4 * j + 2], (float)((w >> 16) & 0xffu), total);
                total = fmaf(xr[4 * j + 3], (float)(w >> 24), total);
            }
            acc[r] = scale * (total - 128.0f * xsum);
        }
        rg += stride;
        __builtin_amdgcn_sched_barrier(0);  // the next loads reuse this tile's registers: keep them behind the arithmetic
        float sum = fold_rows<R, G>(acc, lane);  // lane u < R holds row first + u
        if (rg < p.row_groups) load(held, rg);
        if (DEEP) {
            if (u < R) part[parity][wave][u] = sum;
            __syncthreads();  // every wave walks the same passes
            if (u < R) sum = (part[parity][0][u] + part[parity][1][u]) + (part[parity][2][u] + part[parity][3][u]);
            parity ^= 1u;
            if (wave != 0) continue;
        }
        const uint32_t i = first + u;
        if (p.swiglu) {
            const float up = dpp<DPP_QUAD_XOR1>(sum);
            if (u < R && !(u & 1u) && i + 1 < p.N) p.y[i >> 1] = silu(sum) * up;
        } else if (ROPE) {
            rotate_and_store<R>(p, sum, i, u);
        } else if (u < R && i < p.N) {
            p.y[i] = p.residual ? p.residual[i] + sum : sum;
        }
    }
}

// ------------------------------------------------------------ Q6_K, Q5_K, Q3_K -------
//
// 210-, 176- and 110-byte super-blocks; the first and the last leave rows on 2-byte boundaries.  A wave copies the two
// rows it is about to walk into LDS with aligned 128-bit loads -- a row is contiguous, the copy fully coalesced -- and its
// lanes pick the fields out of LDS.  A lane takes 32 weights of a super-block: eight neighbouring elements
// (8j .. 8j + 7) of each of the four 32-element runs of one half.  In all three formats those share one or two 8-byte
// pieces of low bits and one of high bits, and each run has one scale for the eight:
//   Q6_K (crates/neura-precision/src/ggml.rs:394-407, crates/neura-kernel/src/dot.rs:663-797): (d * scale) * (code - 32)
//   Q5_K (ggml.rs:321-335, dot.rs:621-661): d * sc * code - dmin * m
//   Q3_K (ggml.rs:291-306, dot.rs:544-581): (d * (scale - 32)) * (code - 4), the third bit being the code's top bit
// Every run contributes weight * (sum(x * code) - offset * sum(x)) - minimum * sum(x): the stored codes convert to fp32
// with one instruction each, and sum(x) per eight activations is worked out once per workgroup.  The sums run in lane
// order, not in the reference's run order.
__device__ __forceinline__ uint32_t byte_of(uint32_t word, uint32_t at) { return (word >> (8u * at)) & 0xffu; }

template <int ELEMENT>
struct Staged;

template <>
struct Staged<NH_Q6_K> {
    static constexpr uint32_t BYTES = 210u;
    static constexpr float OFFSET = 32.0f;
    static constexpr bool FLOORS = false;
    // codes[g][h]: elements 8j + 4h .. + 3 of run g, one code a byte
    template <typename Word>
    static __device__ __forceinline__ void unit(const uint8_t *block, Word word, uint32_t half, uint32_t j, uint32_t (&codes)[4][2], float (&weight)[4],
                                                float (&floor)[4]) {
        const float d = half_to_float(*reinterpret_cast<const uint16_t *>(block + 208u));
        const uint32_t scales[2] = {word(192u + half * 8u), word(196u + half * 8u)};  // run g, elements 16c ..: byte 2g + c
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t lows = word(half * 64u + 8u * j + 4u * h), highs = word(half * 64u + 32u + 8u * j + 4u * h);
            const uint32_t pairs = word(128u + half * 32u + 8u * j + 4u * h);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint32_t nibbles = ((g & 1) ? highs : lows) >> (g >= 2 ? 4 : 0);
                codes[g][h] = (nibbles & 0x0f0f0f0fu) | (((pairs >> (2 * g)) & 0x03030303u) << 4);
            }
        }
#pragma unroll
        for (int g = 0; g < 4; g++) {
            weight[g] = d * (float)(int8_t)byte_of(scales[g >> 1], 2u * (g & 1) + (j >> 1));
            floor[g] = 0.0f;
        }
    }
};

template <>
struct Staged<NH_Q5_K> {
    static constexpr uint32_t BYTES = 176u;
    static constexpr float OFFSET = 0.0f;
    static constexpr bool FLOORS = true;
    template <typename Word>
    static __device__ __forceinline__ void unit(const uint8_t *block, Word word, uint32_t half, uint32_t j, uint32_t (&codes)[4][2], float (&weight)[4],
                                                float (&floor)[4]) {
        // runs 0..3 of a half are sub-blocks 4 half + t: nibble group 2 half + t / 2, low nibbles for even t
        const uint32_t header = word(0u);
        const float d = half_to_float((uint16_t)header), dmin = half_to_float((uint16_t)(header >> 16));
        const uint32_t s0 = word(4u), s1 = word(8u), s2 = word(12u);  // the twelve scale bytes (ggml.rs:127-136)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t first = word(48u + half * 64u + 8u * j + 4u * h), second = word(48u + half * 64u + 32u + 8u * j + 4u * h);
            const uint32_t fifths = word(16u + 8u * j + 4u * h);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const uint32_t nibbles = ((t & 2) ? second : first) >> ((t & 1) ? 4 : 0);
                codes[t][h] = (nibbles & 0x0f0f0f0fu) | (((fifths >> (4u * half + t)) & 0x01010101u) << 4);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t a = byte_of(s0, t), b = byte_of(s1, t), c = byte_of(s2, t);
            const uint32_t sc = half ? ((c & 15u) | ((a >> 6) << 4)) : (a & 63u);
            const uint32_t mn = half ? ((c >> 4) | ((b >> 6) << 4)) : (b & 63u);
            weight[t] = d * (float)sc;
            floor[t] = dmin * (float)mn;
        }
    }
};

template <>
struct Staged<NH_Q3_K> {
    static constexpr uint32_t BYTES = 110u;
    static constexpr float OFFSET = 4.0f;
    static constexpr bool FLOORS = false;
    template <typename Word>
    static __device__ __forceinline__ void unit(const uint8_t *block, Word word, uint32_t half, uint32_t j, uint32_t (&codes)[4][2], float (&weight)[4],
                                                float (&floor)[4]) {
        const float d = half_to_float(*reinterpret_cast<const uint16_t *>(block + 108u));
        const uint32_t lows[2] = {word(96u), word(100u)}, highs = word(104u);  // six-bit scales (ggml.rs:224-229)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t pairs = word(32u + half * 32u + 8u * j + 4u * h), thirds = word(8u * j + 4u * h);
#pragma unroll
            for (int t = 0; t < 4; t++) codes[t][h] = ((pairs >> (2 * t)) & 0x03030303u) | (((thirds >> (4u * half + t)) & 0x01010101u) << 2);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            // scale 8 half + 2t + c, c = 1 for elements 16 .. 31 of the run: a nibble of byte 2t + c, two bits of byte 8 + (2t + c) % 4
            const uint32_t at = 2u * (t & 1) + (j >> 1);
            const uint32_t low = byte_of(lows[t >> 1], at);
            const uint32_t nibble = half ? (low >> 4) : (low & 15u);
            const uint32_t top = (byte_of(highs, at) >> (2u * (2u * half + (t >> 1)))) & 3u;
            weight[t] = d * ((float)(nibble | (top << 4)) - 32.0f);
            floor[t] = 0.0f;
        }
    }
};

__device__ __forceinline__ uint32_t skew128(uint32_t i) { return i + (i >> 7) * 4; }

// sixteen bytes from `at`, those at and past `end` read as zero without being touched.  Out of line: only the last rows of a
// tensor come here, and the byte loads would otherwise sit in every caller's loop.
__device__ __noinline__ u32x4 piece_before(const uint8_t *at, const uint8_t *end) {
    uint32_t words[4] = {0u, 0u, 0u, 0u};
    for (uint32_t j = 0; j < 16u; j++)
        if (at + j < end) words[j >> 2] |= (uint32_t)at[j] << (8u * (j & 3u));
    u32x4 held = {words[0], words[1], words[2], words[3]};
    return held;
}

template <int ELEMENT, int RB>
__global__ __launch_bounds__(256) void gemv_staged_kernel(GEMV_LEAD_PARAMETERS) {
    GEMV_TAKE_LEAD;
    typedef Staged<ELEMENT> Format;
    extern __shared__ float xs[];  // [RB][slice]; the sums per eight activations; then the raw row slices, two per wave
    __shared__ float red[256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t split = blockIdx.y;
    const uint32_t blk0 = split * p.blocks_per_split;
    const uint32_t nb = min(p.blocks_per_split, p.nblk - blk0);
    const uint32_t k0 = blk0 * 256u, kn = nb * 256u;
    const uint32_t append_cursor = RB == 1 && p.append_value ? p.rope_cursor[0] : 0u;  // asked for here, wanted at the very end
    // the 16-byte pieces of the two rows `first`, `first + 1` this lane copies: fetched one pair of rows ahead, so the copy
    // of the next pair is in flight while this pair is multiplied (a slice is at most 16 blocks: four pieces a lane and row)
    typedef const __attribute__((address_space(1))) u32x4 *global_uint4;
    u32x4 ahead[2][4];
    uint32_t ahead_lead[2] = {0u, 0u};
    auto fetch = [&](uint32_t first) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const uint32_t i = min(first + r, p.N - 1u);
            const uint8_t *matrix_end;
            const uint8_t *src = row_start(p, weight_row(i, p.N, p.swiglu), matrix_end) + (size_t)blk0 * Format::BYTES;
            ahead_lead[r] = (uint32_t)((uintptr_t)src & 15u);
            const uint8_t *from = src - ahead_lead[r];
            const uint32_t bytes = ahead_lead[r] + nb * Format::BYTES;
            const uint32_t pieces = (bytes + 15u) / 16u;
            if (from + 16u * pieces <= matrix_end) {  // the same for every lane of the wave
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t c = lane + 64u * k;
                    u32x4 held = {0u, 0u, 0u, 0u};
                    if (c < pieces) held = *(global_uint4)(uintptr_t)(from + 16u * c);
                    ahead[r][k] = held;
                }
            } else {  // the last bytes of the tensor: never read past its end
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t c = lane + 64u * k;
                    u32x4 held = {0u, 0u, 0u, 0u};
                    if (c < pieces) held = piece_before(from + 16u * c, matrix_end);
                    ahead[r][k] = held;
                }
            }
        }
    };
    const uint32_t stride = 2u * gridDim.x * 4u;
    uint32_t first = 2u * (blockIdx.x * 4u + wave);
    if (first < p.N) fetch(first);  // on its way while the activations are staged
    // halves of 128 activations sit 16 bytes apart: the lanes of a wave read eight of them at once
    const uint32_t xstride = skew128(p.blocks_per_split * 256u);
    for (uint32_t b = 0; b < RB; b++) {
        stage_row(p.x + (size_t)b * p.K, p.K, k0, kn, p.norm_w, p.eps, xs + b * xstride, red, [](uint32_t i) { return skew128(i); });
    }
    __syncthreads();
    // what the codes' offset (or a run's minimum) multiplies, once for all rows: per unit and run the sum of the eight
    // activations, times the offset where the format has one
    float *const sums = xs + RB * xstride;
    const uint32_t sstride = p.blocks_per_split * 32u;
    for (uint32_t b = 0; b < RB; b++)
        for (uint32_t q = tid; q < nb * 32u; q += 256u) {
            const uint32_t u = q >> 2, g = q & 3u;
            const float4 *at = reinterpret_cast<const float4 *>(xs + b * xstride + skew128((u >> 2) * 128u) + g * 32u + 8u * (u & 3u));
            const float4 lo = at[0], hi = at[1];
            const float total = ((lo.x + lo.y) + (lo.z + lo.w)) + ((hi.x + hi.y) + (hi.z + hi.w));
            sums[b * sstride + q] = Format::FLOORS ? total : -Format::OFFSET * total;
        }
    __syncthreads();
    const uint32_t raw_stride = p.chunks_per_row * 16u;  // bytes of one staged row slice
    uint8_t *const mine = reinterpret_cast<uint8_t *>(sums + RB * sstride) + (size_t)wave * 2u * raw_stride;
    const uint32_t units = nb * 8u;

    for (; first < p.N; first += stride) {
        uint32_t lead[2];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            lead[r] = ahead_lead[r];
#pragma unroll
            for (int k = 0; k < 4; k++)
                if ((lane + 64u * k) < p.chunks_per_row) *reinterpret_cast<u32x4 *>(mine + r * raw_stride + 16u * (lane + 64u * k)) = ahead[r][k];
        }
        if (first + stride < p.N) fetch(first + stride);
        __builtin_amdgcn_wave_barrier();  // LDS serves a wave's accesses in order: the reads below see these writes

        float acc[2][RB];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int b = 0; b < RB; b++) acc[r][b] = 0.0f;
        for (uint32_t u = lane; u < units; u += 64u) {
            const uint32_t blk = u >> 3, half = (u >> 2) & 1u, j = u & 3u;
            float4 xv[RB][4][2];
            float base[RB][4];
#pragma unroll
            for (int b = 0; b < RB; b++) {
                const float4 held = *reinterpret_cast<const float4 *>(sums + b * sstride + 4u * u);
                base[b][0] = held.x, base[b][1] = held.y, base[b][2] = held.z, base[b][3] = held.w;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float4 *at = reinterpret_cast<const float4 *>(xs + b * xstride + skew128(blk * 256u + half * 128u) + g * 32u + 8u * j);
                    xv[b][g][0] = at[0], xv[b][g][1] = at[1];
                }
            }
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const uint8_t *block = mine + r * raw_stride + lead[r] + blk * Format::BYTES;
                // a block sits on a 2-byte boundary: its words are cut out of the aligned words around them (LDS serves a
                // misaligned read at a fraction of its rate)
                const uint32_t off = Format::BYTES % 4u ? (uint32_t)(uintptr_t)block & 3u : 0u;
                const uint32_t *words = reinterpret_cast<const uint32_t *>(block - off);
                auto word = [&](uint32_t at) {
                    if (Format::BYTES % 4u == 0) return words[at / 4u];
                    return __builtin_amdgcn_alignbit(words[at / 4u + 1u], words[at / 4u], off * 8u);
                };
                uint32_t codes[4][2];
                float weight[4], floor[4];
                Format::unit(block, word, half, j, codes, weight, floor);
#pragma unroll
                for (int g = 0; g < 4; g++) {
#pragma unroll
                    for (int b = 0; b < RB; b++) {
                        // the codes go to fp32 as they are stored, one conversion each; their offset came with the sum
                        float dot = Format::FLOORS ? 0.0f : base[b][g];
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const uint32_t c = codes[g][h];
                            dot = fmaf(xv[b][g][h].x, (float)(c & 0xffu), dot);
                            dot = fmaf(xv[b][g][h].y, (float)((c >> 8) & 0xffu), dot);
                            dot = fmaf(xv[b][g][h].z, (float)((c >> 16) & 0xffu), dot);
                            dot = fmaf(xv[b][g][h].w, (float)(c >> 24), dot);
                        }
                        acc[r][b] = fmaf(weight[g], dot, acc[r][b]);
                        if (Format::FLOORS) acc[r][b] = fmaf(-floor[g], base[b][g], acc[r][b]);
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int b = 0; b < RB; b++) acc[r][b] = wave_sum(acc[r][b]);
        if (lane == 0) publish<2, RB>(p, first, split, acc);
        if (RB == 1 && p.append_value && lane < 2 && first + lane < p.N) {
            // a value projection of one token: its rows (+ bias) go into the value state at the cursor as halves, as
            // value_append_kernel would cast them
            const uint32_t n = first + lane;
            const float sum = lane ? acc[1][0] : acc[0][0];
            const float value = p.bias[0] ? sum + p.bias[0][n] : sum;
            const uint32_t slot = p.rope_ring ? append_cursor % p.rope_ring : append_cursor;
            if (slot >= p.rope_capacity) atomicMax(p.refusal, (uint32_t)REFUSAL_ORIGIN);
            else state_store(p.rope_v, p.rope_element, ((uint64_t)(n / p.rope_width) * p.rope_capacity + slot) * p.rope_width + n % p.rope_width, value);
        }
        __builtin_amdgcn_wave_barrier();  // the next rows overwrite the staged ones
    }
}

// ------------------------------------------------------------------------- fold ----------

// sums the slice partials in slice order and applies the epilogue
// (crates/neura-kernel/src/task/matmul.rs:1318-1333)
__global__ __launch_bounds__(256) void gemv_fold_kernel(const float *__restrict__ partial, uint32_t splits, uint32_t rows, uint32_t N,
                                                        const float *__restrict__ residual, int32_t swiglu, float *__restrict__ y) {
    NH_FETCH(partial, splits, rows, N, residual, swiglu, y, blockDim.x);
    uint32_t outputs = swiglu ? N / 2 : N;
    for (uint32_t index = blockIdx.x * blockDim.x + threadIdx.x; index < rows * outputs; index += gridDim.x * blockDim.x) {
        uint32_t b = index / outputs, n = index % outputs;
        // eight slices at a time, every load asked for before the first is added (past the last slice the last again,
        // dropped): the sum still runs in slice order
        auto sum_of = [&](uint32_t column) {
            float total = 0.0f;
            for (uint32_t s0 = 0; s0 < splits; s0 += 8u) {
                float held[8];
#pragma unroll
                for (int j = 0; j < 8; j++) held[j] = partial[((size_t)min(s0 + j, splits - 1u) * rows + b) * N + column];
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (s0 + j < splits) total += held[j];
            }
            return total;
        };
        float total = sum_of(n);
        if (swiglu) {
            const float up = sum_of(N / 2 + n);
            total = silu(total) * up;
        } else if (residual) {
            total = residual[(size_t)b * N + n] + total;
        }
        y[(size_t)b * outputs + n] = total;
    }
}

// ------------------------------------------------------------------------- host ----------

static uint32_t pow2_at_least(uint32_t v, uint32_t floor) {
    uint32_t p = floor;
    while (p < v) p <<= 1;
    return p;
}


template <int RB>
static int32_t launch_rows(nh_device *d, const GemvArgs &a, const float *x, float *y, const float *residual) {
    GemvParams p{};
    for (int s = 0; s < 3; s++) {
        p.W[s] = static_cast<const uint8_t *>(a.W[s] ? a.W[s] : a.W[0]);
        p.end[s] = a.end[s];
    }
    p.x = x;
    if (a.merge) p.x = a.merge->partial, p.merge_sections = a.merge->sections, p.merge_groups = a.merge->groups, p.merge_width = a.merge->width;
    p.y = y;
    p.residual = residual;
    p.norm_w = a.norm_w;
    p.N = a.N;
    p.K = a.K;
    p.swiglu = a.swiglu;
    p.eps = a.eps;
    if (a.rope) {
        p.rope_cosines = a.rope->cosines, p.rope_sines = a.rope->sines, p.rope_cursor = a.rope->cursor, p.rope_k = a.rope->cache_k, p.rope_v = a.rope->cache_v;
        p.rope_width = a.rope->width, p.rope_q_rows = a.rope->q_rows, p.rope_k_rows = a.rope->k_rows, p.rope_capacity = a.rope->capacity;
        p.rope_positions = a.rope->positions, p.rope_ring = a.rope->ring, p.rope_element = a.rope->element;
        p.refusal = d->refusal;
        for (int s = 0; s < 3; s++) p.bias[s] = a.bias[s];
    } else if (a.bias[0] || a.bias[1] || a.bias[2]) {
        return fail(NH_E_ARGUMENT, "a product adds a bias only where it folds the rotation in");
    }
    p.row_bytes = (uint32_t)payload_bytes(a.element, a.K);
    const bool q4 = a.element == NH_Q4_K;
    p.nblk = a.K / (q4 ? 256u : 32u);
    // one lane per 64 (Q4_K) or 32 (Q8_0) elements; a slice fills at most one wave
    uint32_t units_per_block = q4 ? 4u : 1u;
    uint32_t most_blocks = q4 ? (RB >= 4 ? 8u : 16u) : 64u;
    p.splits = (p.nblk + most_blocks - 1) / most_blocks;
    p.blocks_per_split = (p.nblk + p.splits - 1) / p.splits;
    p.splits = (p.nblk + p.blocks_per_split - 1) / p.blocks_per_split;
    p.group = pow2_at_least(p.blocks_per_split * units_per_block, 16u);
    uint32_t RS = 64u / p.group;
    if (p.splits > 1) {
        p.partial = static_cast<float *>(scratch(d, (size_t)p.splits * RB * a.N * sizeof(float)));
        if (!p.partial) return NH_E_MEMORY;
    }
    // rows per lane group and pass: four rows amortise the cross-lane sum and keep more bytes
    // in flight per wave, two rows give twice the waves; tall matrices take four
    int R = (a.N >= 16384u && RB == 1) ? 4 : 2;
    if (RB >= 4) R = 2;
    // the decode kernel walks R rows of ONE matrix per lane group: every matrix boundary must be a
    // multiple of R (with swiglu the halves interleave, so N/2 must be a multiple of R/2)
    auto whole = [&](int rows) {
        if (a.swiglu) return a.N % (uint32_t)rows == 0 && a.end[0] == a.N / 2;
        return a.end[0] % (uint32_t)rows == 0 && a.end[1] % (uint32_t)rows == 0 && a.N % (uint32_t)rows == 0;
    };
    if (R == 4 && !whole(4)) R = 2;
    const bool fast = whole(R) && a.N >= (uint32_t)R && (uint64_t)a.N * p.row_bytes < (1ull << 32);
    uint32_t rows_per_pass = (uint32_t)R * RS;
    p.row_groups = (a.N + rows_per_pass - 1) / rows_per_pass;
    uint32_t blocks_x;
    size_t lds;
    if (q4) {
        blocks_x = (p.row_groups + 3) / 4;
        // one resident round of workgroups: 3 per compute unit at four rows (136 registers), 4 at two
        uint32_t most = (uint32_t)d->compute_units * (R == 4 ? 3u : 4u) / p.splits;
        if (most < 1) most = 1;
        if (blocks_x > most) blocks_x = most;
        uint32_t slice = p.blocks_per_split * 256u;
        lds = (size_t)RB * (slice + slice / 64 * 4) * sizeof(float);
    } else {
        uint32_t slice_bytes = p.blocks_per_split * 34u;
        p.chunks_per_row = (15u + slice_bytes + 15u) / 16u;
        uint32_t tiles = (p.row_groups + 3) / 4;
        blocks_x = tiles;
        uint32_t most = (uint32_t)d->compute_units * 4u / p.splits;
        if (most < 1) most = 1;
        if (blocks_x > most) blocks_x = most;
        uint32_t slice = p.blocks_per_split * 32u;
        lds = (size_t)RB * (slice + slice / 32 * 4) * sizeof(float) + (size_t)rows_per_pass * 4 * p.chunks_per_row * 16 + 16;
    }
    if (lds > 64 * 1024) return fail(NH_E_ARGUMENT, "a product of depth %u stages %zu bytes where a workgroup holds 65536", a.K, lds);
    dim3 grid(blocks_x, p.splits), block(256);
    profile_mark(d);
#define NH_LAUNCH(KERNEL, RR) hipLaunchKernelGGL((KERNEL<RR, RB>), grid, block, lds, d->stream, p)
#define NH_DECODE(RR, GG) hipLaunchKernelGGL((gemv_q4k_decode_kernel<RR, GG, false, 4>), grid, block, lds, d->stream, p)
    const bool q8_direct = !q4 && RB == 1 && fast && p.nblk <= 256u;
    if (a.merge && !(q8_direct && R == 2 && p.nblk <= 64u && !a.rope))
        return fail(NH_E_ARGUMENT, "this product merges no attention sections (ask gemv_merges_sections first)");
    if (a.rope && !(q4 && RB == 1 && fast && R == 2 && p.splits == 1) && !(q8_direct && R == 2 && p.nblk <= 64u))
        return fail(NH_E_ARGUMENT, "this product cannot fold the rotation in (ask gemv_fuses_rope first)");
    if (q4 && RB == 1 && fast && a.rope) {
        if (p.group == 64) hipLaunchKernelGGL((gemv_q4k_decode_kernel<2, 64, false, 4, true>), grid, block, lds, d->stream, p);
        else if (p.group == 32) hipLaunchKernelGGL((gemv_q4k_decode_kernel<2, 32, false, 4, true>), grid, block, lds, d->stream, p);
        else hipLaunchKernelGGL((gemv_q4k_decode_kernel<2, 16, false, 4, true>), grid, block, lds, d->stream, p);
    } else if (q4 && RB == 1 && fast) {
        if (R == 4) {
            if (p.group == 64) NH_DECODE(4, 64);
            else if (p.group == 32) NH_DECODE(4, 32);
            else NH_DECODE(4, 16);
        } else {
            if (p.group == 64) NH_DECODE(2, 64);
            else if (p.group == 32) NH_DECODE(2, 32);
            else NH_DECODE(2, 16);
        }
    } else if (q4) {
        if (R == 4) NH_LAUNCH(gemv_q4k_kernel, 4);
        else NH_LAUNCH(gemv_q4k_kernel, 2);
    } else if (q8_direct) {
        // one activation row, a row of blocks inside one wave (or, deeper, inside the four waves of a workgroup): the words of
        // a block straight from memory, no LDS tile, no K slices and no fold
        const bool deep = p.nblk > 64u;
        if (deep) p.group = 64, RS = 1;
        p.splits = 1, p.blocks_per_split = p.nblk;
        const uint32_t passes = (a.N + (uint32_t)R * RS - 1) / ((uint32_t)R * RS);
        p.row_groups = passes;
        uint32_t wgs = deep ? passes : (passes + 3) / 4;
        const uint32_t resident = (uint32_t)d->compute_units * 4u;
        if (wgs > resident) wgs = resident;
        const size_t staged = (size_t)(a.K + a.K / 32u * 4u) * sizeof(float);
        const dim3 wide(wgs);
#define NH_Q8(RR, GG) hipLaunchKernelGGL((gemv_q8_0_decode_kernel<RR, GG>), wide, block, staged, d->stream, Q8_LEAD(p))
        if (a.rope) {
            if (p.group == 64) hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 64, false, true>), wide, block, staged, d->stream, Q8_LEAD(p));
            else if (p.group == 32) hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 32, false, true>), wide, block, staged, d->stream, Q8_LEAD(p));
            else hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 16, false, true>), wide, block, staged, d->stream, Q8_LEAD(p));
        } else if (a.merge) {
            if (p.group == 64) hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 64, false, false, true>), wide, block, staged, d->stream, Q8_LEAD(p));
            else if (p.group == 32) hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 32, false, false, true>), wide, block, staged, d->stream, Q8_LEAD(p));
            else hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 16, false, false, true>), wide, block, staged, d->stream, Q8_LEAD(p));
        } else if (deep) {
            if (R == 4) hipLaunchKernelGGL((gemv_q8_0_decode_kernel<4, 64, true>), wide, block, staged, d->stream, Q8_LEAD(p));
            else hipLaunchKernelGGL((gemv_q8_0_decode_kernel<2, 64, true>), wide, block, staged, d->stream, Q8_LEAD(p));
        } else if (R == 4) {
            if (p.group == 64) NH_Q8(4, 64);
            else if (p.group == 32) NH_Q8(4, 32);
            else NH_Q8(4, 16);
        } else {
            if (p.group == 64) NH_Q8(2, 64);
            else if (p.group == 32) NH_Q8(2, 32);
            else NH_Q8(2, 16);
        }
#undef NH_Q8
    } else {
        if (R == 4) NH_LAUNCH(gemv_q8_0_kernel, 4);
        else NH_LAUNCH(gemv_q8_0_kernel, 2);
    }
#undef NH_LAUNCH
#undef NH_DECODE
    NH_HIP(hipGetLastError());
    if (p.splits > 1) {
        uint32_t outputs = (a.swiglu ? a.N / 2 : a.N) * RB;
        hipLaunchKernelGGL(gemv_fold_kernel, dim3((outputs + 255) / 256), dim3(256), 0, d->stream, p.partial, p.splits, (uint32_t)RB, a.N,
                           residual, a.swiglu, y);
        NH_HIP(hipGetLastError());
    }
    profile_mark(d);
    if (d->profile) d->profile_bytes += (uint64_t)a.N * p.row_bytes;
    return NH_OK;
}

// mirrors the conditions under which launch_rows<1> takes the decode kernel with two rows per pass
bool gemv_fuses_rope(const GemvArgs &a, const RopeFusion &rope) {
    if (env_int("NEURA_HIP_FUSE_ROPE", 1) == 0) return false;
    if (a.rows > 1) {  // one token of each of several planes
        GemvArgs folded = a;
        folded.rope = &rope;
        return rows_takes(folded);
    }
    if (a.rows != 1 || a.swiglu || a.residual) return false;
    {
        GemvArgs folded = a;
        folded.rope = &rope;
        if (tile16_takes(folded) || q6k_tile16_takes(folded)) return true;
    }
    if (a.element == NH_Q8_0) {
        // the direct Q8_0 decode kernel, a row of blocks inside one wave
        if (a.K % 32u != 0 || a.K > 2048u ) return false;
        if (a.N >= 16384u || a.N < 2u || (uint64_t)a.N * (a.K / 32u * 34u) >= (1ull << 32)) return false;
        if (a.end[0] % 2u || a.end[1] % 2u || a.N % 2u) return false;
    } else {
        if (a.element != NH_Q4_K || a.K % 256u != 0 || a.K > 4096u) return false;
        if (a.N >= 16384u || a.N < 2u || (uint64_t)a.N * (a.K / 256u * 144u) >= (1ull << 32)) return false;
    }
    const uint32_t width = rope.width;
    if (width < 2 || (width & (width - 1u)) != 0) return false;
    if (rope.q_rows % width || rope.k_rows % width || a.N % width || rope.q_rows > rope.k_rows || rope.k_rows > a.N) return false;
    // a head never straddles two matrices
    return a.end[0] % width == 0 && a.end[1] % width == 0 && a.end[2] == a.N;
}

// Q6_K, Q5_K, Q3_K: one, two or four activation rows a launch (their slices and the raw rows share LDS: three workgroups a compute unit)
template <int ELEMENT, int RB>
static int32_t launch_staged_rows(nh_device *d, const GemvArgs &a, const float *x, float *y, const float *residual) {
    GemvParams p{};
    for (int s = 0; s < 3; s++) {
        p.W[s] = static_cast<const uint8_t *>(a.W[s] ? a.W[s] : a.W[0]);
        p.end[s] = a.end[s];
    }
    p.x = x, p.y = y, p.residual = residual, p.norm_w = a.norm_w;
    p.N = a.N, p.K = a.K, p.swiglu = a.swiglu, p.eps = a.eps;
    p.row_bytes = (uint32_t)payload_bytes(ELEMENT, a.K);
    p.nblk = a.K / 256u;
    if (a.append_value) {
        if (RB != 1 || a.swiglu || residual || p.nblk > 16u || !a.append_value->width || a.N % a.append_value->width)
            return fail(NH_E_ARGUMENT, "this product appends no value rows (one row, one K slice, whole heads, no other epilogue)");
        p.append_value = 1u, p.rope_v = a.append_value->cache_v, p.rope_cursor = a.append_value->cursor, p.rope_width = a.append_value->width;
        p.rope_capacity = a.append_value->capacity, p.rope_ring = a.append_value->ring, p.rope_element = a.append_value->element, p.bias[0] = a.bias[0], p.refusal = d->refusal;
    }
    // K slices of sixteen super-blocks at most; of eight with four activation rows, whose slices take the room of two rows' twice over
    const uint32_t most_blocks = RB == 4 ? 8u : 16u;
    p.splits = (p.nblk + most_blocks - 1) / most_blocks;
    p.blocks_per_split = (p.nblk + p.splits - 1) / p.splits;
    p.splits = (p.nblk + p.blocks_per_split - 1) / p.blocks_per_split;
    if (p.splits > 1) {
        p.partial = static_cast<float *>(scratch(d, (size_t)p.splits * RB * a.N * sizeof(float)));
        if (!p.partial) return NH_E_MEMORY;
    }
    p.chunks_per_row = (15u + p.blocks_per_split * Staged<ELEMENT>::BYTES + 15u) / 16u + 1u;  // a lead, the blocks, and the word past the last field
    // activation slices (8 floats of skew a block), their sums per eight, the raw rows
    const size_t lds = (size_t)RB * p.blocks_per_split * (264u + 32u) * sizeof(float) + (size_t)8 * p.chunks_per_row * 16u;
    uint32_t blocks_x = (a.N + 7u) / 8u;
    // three workgroups a compute unit: their LDS (about 41 KiB each at 14 blocks) and registers fit, and a fourth measured slower
    uint32_t most = (uint32_t)d->compute_units * 3u / p.splits;
    if (most < 1) most = 1;
    if (blocks_x > most) blocks_x = most;
    profile_mark(d);
    if (lds > 64u * 1024u) {
        static OnceADevice widened;  // past 64 KiB of dynamic LDS a kernel has to be told
        NH_HIP(raise_lds(widened, d, reinterpret_cast<const void *>(&gemv_staged_kernel<ELEMENT, RB>), 158 * 1024));
    }
    hipLaunchKernelGGL((gemv_staged_kernel<ELEMENT, RB>), dim3(blocks_x, p.splits), dim3(256), lds, d->stream, GEMV_LEAD(p));
    NH_HIP(hipGetLastError());
    if (p.splits > 1) {
        uint32_t outputs = (a.swiglu ? a.N / 2 : a.N) * RB;
        hipLaunchKernelGGL(gemv_fold_kernel, dim3((outputs + 255) / 256), dim3(256), 0, d->stream, p.partial, p.splits, (uint32_t)RB, a.N,
                           residual, a.swiglu, y);
        NH_HIP(hipGetLastError());
    }
    profile_mark(d);
    if (d->profile) d->profile_bytes += (uint64_t)a.N * p.row_bytes;
    return NH_OK;
}

// What the Q8_0 decode kernel of two rows a lane group takes (launch_rows<1> sends such a product there), and the merge's own
// bounds: whole heads, no more of them than the statistics' corner of LDS holds.
bool gemv_merges_sections(const GemvArgs &a, uint32_t width) {
    if (!env_int("NEURA_HIP_MERGE_IN_PRODUCT", 1) || a.element != NH_Q8_0 || a.rows != 1 || a.rope || a.swiglu || a.norm_w || a.digits_in || a.digits_out) return false;
    if (!width || (width & (width - 1u)) || a.K % 32u || a.K / 32u > 64u || a.K % width || a.K / width > 32u) return false;
    if (a.N < 2u || a.N >= 16384u || a.N % 2u || a.end[0] % 2u || a.end[1] % 2u) return false;
    return (uint64_t)a.N * payload_bytes(a.element, a.K) < (1ull << 32);
}

// Whether a product with `append_value` set casts its rows into the value state itself: one row of a K-quant on the 16-row
// tiles, or on the staged kernel where a row is one K slice.
bool gemv_appends_value(const GemvArgs &a) {
    if (!a.append_value || a.rows != 1 || a.rope || a.swiglu || a.residual) return false;
    if (tile16_takes(a) || q6k_tile16_takes(a)) return true;
    return staged_super_block(a.element) && a.K <= 4096u && a.append_value->width && a.N % a.append_value->width == 0;
}

// (past 1792 numbers the norm's scalar would be the fold's and the rotation a kernel of its own: not the line yet, though the 7B shape at nine planes
// takes 2.82 ms a step in place of 3.21 without it, and rows of 2048 numbers 1.16 in place of 1.23)
bool gemv_takes_many(const GemvArgs &a) { return a.rows > 8 && (!a.norm_w || a.K <= 1792u) && rows_takes(a); }

// (the vector and staged forms walk four rows at most at a time, in slices of 2048 numbers at least)
size_t gemv_scratch_bytes(uint32_t N, uint32_t K, uint32_t rows) {
    size_t most = K > 2048u ? (size_t)((K + 2047u) / 2048u) * min(rows, 4u) * N * sizeof(float) : 0u;
    for (uint32_t r = 2; r <= min(rows, 16u) && K % 256u == 0; r++) most = max(most, rows_scratch_bytes(N, K, r));
    return most;
}

int32_t launch_gemv(nh_device *d, const GemvArgs &a) {
    if (!a.rope && !a.append_value && (a.bias[0] || a.bias[1] || a.bias[2]))
        return fail(NH_E_ARGUMENT, "a product adds a bias only where it folds the rotation in or appends value rows");
    if (a.append_value && !gemv_appends_value(a))
        return fail(NH_E_ARGUMENT, "this product does not append its rows to the value state (ask gemv_appends_value first)");
    if (a.merge && (!gemv_merges_sections(a, a.merge->width) || a.merge->sections < 2u || a.merge->sections > MERGED_SECTIONS_MOST || !a.merge->groups ||
                    (a.K / a.merge->width) % a.merge->groups))
        return fail(NH_E_ARGUMENT, "this product merges no attention sections (ask gemv_merges_sections first)");
    if (a.merge) return launch_rows<1>(d, a, a.x, a.y, a.residual);
    if (a.rows > 2 && rows_takes(a)) return launch_q4k_rows(d, a);
    if (tile16_takes(a)) return launch_tile16(d, a);
    if (q6k_tile16_takes(a)) return launch_q6k_tile16(d, a);
    if (a.digits_out || a.digits_in) return fail(NH_E_ARGUMENT, "this product hands over no digit planes (ask gemv_hands_digits first)");
    if (a.rope && a.rows != 1) return fail(NH_E_ARGUMENT, "this product cannot fold the rotation in (ask gemv_fuses_rope first)");
    if (rows_takes(a)) return launch_q4k_rows(d, a);
    if (gemv_wide_takes(d, a)) return launch_gemv_wide(d, a);
    // activation rows are taken four, two or one at a time
    uint32_t outputs = a.swiglu ? a.N / 2 : a.N;
    uint32_t done = 0;
    if (staged_super_block(a.element)) {
        if (a.swiglu && (a.N % 2u || a.end[0] != a.N / 2)) return fail(NH_E_ARGUMENT, "a swiglu product halves %u rows", a.N);
        while (done < a.rows) {
            const float *x = a.x + (size_t)done * a.K;
            float *y = a.y + (size_t)done * outputs;
            const float *residual = a.residual ? a.residual + (size_t)done * a.N : nullptr;
            const bool pair = a.rows - done >= 2;
            const bool four = a.rows - done >= 4;  // (Q6_K 512 x 3584: 9.5 us, two rows a pass twice 7.1)
            int32_t status;
            if (a.element == NH_Q6_K)
                status = four ? launch_staged_rows<NH_Q6_K, 4>(d, a, x, y, residual)
                         : pair ? launch_staged_rows<NH_Q6_K, 2>(d, a, x, y, residual) : launch_staged_rows<NH_Q6_K, 1>(d, a, x, y, residual);
            else if (a.element == NH_Q5_K)
                status = four ? launch_staged_rows<NH_Q5_K, 4>(d, a, x, y, residual)
                         : pair ? launch_staged_rows<NH_Q5_K, 2>(d, a, x, y, residual) : launch_staged_rows<NH_Q5_K, 1>(d, a, x, y, residual);
            else
                status = four ? launch_staged_rows<NH_Q3_K, 4>(d, a, x, y, residual)
                         : pair ? launch_staged_rows<NH_Q3_K, 2>(d, a, x, y, residual) : launch_staged_rows<NH_Q3_K, 1>(d, a, x, y, residual);
            if (status != NH_OK) return status;
            done += four ? 4 : (pair ? 2 : 1);
        }
        return NH_OK;
    }
    while (done < a.rows) {
        uint32_t left = a.rows - done;
        const float *x = a.x + (size_t)done * a.K;
        float *y = a.y + (size_t)done * outputs;
        const float *residual = a.residual ? a.residual + (size_t)done * a.N : nullptr;
        int32_t status;
        if (left >= 4) {
            status = launch_rows<4>(d, a, x, y, residual);
            done += 4;
        } else if (left >= 2) {
            status = launch_rows<2>(d, a, x, y, residual);
            done += 2;
        } else {
            status = launch_rows<1>(d, a, x, y, residual);
            done += 1;
        }
        if (status != NH_OK) return status;
    }
    return NH_OK;
}

}  // namespace nh
