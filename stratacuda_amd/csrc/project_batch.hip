// Dense projections. A token batch (strata_bf16_project and
// strata_quant_project with two or more tokens): every weight is read and
// widened once for up to 16 tokens, with the reference's sums. One token of
// quantized weights: k_project_one below.
//
// The reference's order (kernels/strata.cu:156-165) is 64 partial sums per
// output, partial p over the columns p, p + 64, ... one rounded product and
// one rounded sum at a time, then a tree. The sums have to stay on the vector
// unit, but the products need not: v_mfma_f32_4x4x1_16b_f32 with a zero
// accumulator forms 16 independent 4 x 4 outer products, each element one
// f32 product rounded to nearest even (subnormals kept; an exact -0 becomes
// +0, which a partial sum that starts at +0 cannot tell apart). A block of
// the instruction is one column, its rows four tokens and its columns four
// weight rows, so four of them are the 64 columns of a step and every lane
// then adds its own 4 x 4 products: one matrix instruction for four vector
// adds where the vector unit alone would need four multiplies as well.
//
// A wave owns four weight rows and 4 NG tokens. Lane l holds columns
// 4 (l / 4) .. + 3 of the step's 64 for weight row l % 4, and reads the same
// columns of token 4 g + l % 4 from LDS with one 16-byte load per group of
// four tokens. The block's four waves share the tokens' columns, which
// arrive by DMA one chunk of KC steps ahead; the weights go straight to
// registers one chunk ahead.
//
// Bound: vector issue from about 8 tokens (16 tokens: 64 adds and 16 matrix
// instructions a step; vector instructions issue 57 % of the SIMDs' time, the
// matrix unit is busy 15 %), the weights' stream below (a load's latency per
// chunk, 3 TB/s). bf16, 2,560 x 10,240 x 16 tokens: 208 -> 33 us, where one
// wave per output and token read each weight 16 times. Three or four chunks
// of weights in registers were slower (35 against 31 us in one run: fewer
// waves fit and the loads past the end count).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.h"
#include "strata_device.h"

using namespace smi;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

// The raw weights of one lane and one step: four columns of one row.
template <int BITS>
struct Raw {
    uint32_t code[BITS == 32 ? 4 : BITS == 16 ? 2 : 1];
    float scale, offset;
};

struct ProjectArgs {
    const float *X;
    const uint8_t *codes;
    const float *scales, *offsets;
    float *Y;
    int cols, rows, tokens, stride, out;
    int group_shift, has_offset;
    float bias;
    // the router (f32 weights): its last row and that row's outputs when there
    // is a shared-expert gate, and the experts' biases
    const float *gate_row, *expert_bias;
    float *gate_out;
};

// IQ4_NL values (kernels/strata.cu:22-31) as signed bytes, four to a word.
constexpr uint32_t iq4_word(int a, int b, int c, int d) {
    return (uint32_t)(a & 255) | (uint32_t)(b & 255) << 8 | (uint32_t)(c & 255) << 16 | (uint32_t)(d & 255) << 24;
}

template <int BITS>
__device__ __forceinline__ void load_raw(const ProjectArgs &a, const uint8_t *row_codes, const float *row_scales,
                                         const float *row_offsets, int col, Raw<BITS> &w) {
    if constexpr (BITS == 32) {
        const uint4 v = *(const uint4 *)(row_codes + 4 * col);
        w.code[0] = v.x;
        w.code[1] = v.y;
        w.code[2] = v.z;
        w.code[3] = v.w;
    } else if constexpr (BITS == 16) {
        const uint2 v = *(const uint2 *)(row_codes + 2 * col);
        w.code[0] = v.x;
        w.code[1] = v.y;
    } else {
        if (BITS == 8) w.code[0] = *(const uint32_t *)(row_codes + col);
        if (BITS == 4) w.code[0] = *(const uint16_t *)(row_codes + col / 2);
        if (BITS == 2) w.code[0] = row_codes[col / 4];
        const int g = col >> a.group_shift;
        w.scale = row_scales[g];
        w.offset = row_offsets[g];
    }
}

// The values of four quantized weights, before their scale and offset.
template <int BITS, bool CODEBOOK>
__device__ __forceinline__ void unpack(const ProjectArgs &a, uint32_t c, float (&out)[4]) {
    if (CODEBOOK) {
        // the four codes in four bytes, looked up in the table's two halves
        const uint32_t t = (c | c << 8) & 0x00ff00ffu, b = (t | t << 4) & 0x0f0f0f0fu, s = b & 0x07070707u;
        const uint32_t lo = __builtin_amdgcn_perm(iq4_word(-49, -35, -22, -10), iq4_word(-127, -104, -83, -65), s);
        const uint32_t hi = __builtin_amdgcn_perm(iq4_word(53, 69, 89, 113), iq4_word(1, 13, 25, 38), s);
        const uint32_t m = ((b >> 3) & 0x01010101u) * 255u, v = (hi & m) | (lo & ~m);
#pragma unroll
        for (int q = 0; q < 4; q++) out[q] = (float)((int)(v << (24 - 8 * q)) >> 24);
    } else {
        // code + bias: both are whole numbers below 2^23, so the f32 sum is exact
#pragma unroll
        for (int q = 0; q < 4; q++) out[q] = (float)((c >> (BITS * q)) & ((1u << BITS) - 1u)) + a.bias;
    }
}

// Widens the four weights in the reference's steps (kernels/strata.cu:168-211).
// Without offsets +0 is added: that can only turn a weight of -0 into +0, and
// no partial sum tells a product of -0 from one of +0.
template <int BITS, bool CODEBOOK>
__device__ __forceinline__ void widen(const ProjectArgs &a, const Raw<BITS> &w, float (&out)[4]) {
    if constexpr (BITS == 32) {
#pragma unroll
        for (int q = 0; q < 4; q++) out[q] = __uint_as_float(w.code[q]);
        return;
    } else if constexpr (BITS == 16) {
        out[0] = __uint_as_float(w.code[0] << 16);
        out[1] = __uint_as_float(w.code[0] & 0xffff0000u);
        out[2] = __uint_as_float(w.code[1] << 16);
        out[3] = __uint_as_float(w.code[1] & 0xffff0000u);
        return;
    } else {
        unpack<BITS, CODEBOOK>(a, w.code[0], out);
#pragma unroll
        for (int q = 0; q < 4; q++) out[q] = out[q] * w.scale;
        const float offset = a.has_offset ? w.offset : 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) out[q] = out[q] + offset;
    }
}

// The reference's tree over columns for one group's 4 x 4 products: partial
// sums of column 4 b + q are in lanes 4 b .. 4 b + 3 (one weight row each)
// of p[q], element r for token r. Distances 32, 16, 8 and 4 are lanes 32,
// 16, 8 and 4 apart; 2 and 1 are q. The two lane swaps leave each row of 16
// lanes one token: 0, 2, 1, 3.
__device__ __forceinline__ float tree_columns(const f32x4 (&p)[4]) {
    float z[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        // (__float_as_uint and back: a bit cast of a vector's element takes its first one)
        const auto s01 = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[q][0]), __float_as_uint(p[q][1]), false, false);
        const auto s23 = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[q][2]), __float_as_uint(p[q][3]), false, false);
        const float u = __uint_as_float(s01[0]) + __uint_as_float(s01[1]);
        const float v = __uint_as_float(s23[0]) + __uint_as_float(s23[1]);
        const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(v), false, false);
        float w = __uint_as_float(t[0]) + __uint_as_float(t[1]);
        w = w + sm::dpp_f32<0x108>(0.0f, w);  // row_shl:8
        z[q] = w + sm::dpp_f32<0x104>(0.0f, w);  // row_shl:4
    }
    return (z[0] + z[2]) + (z[1] + z[3]);
}

// Grid: x = groups of 16 weight rows, y = groups of 4 NG tokens. Rows,
// tokens and steps past the end read the last valid one and are not stored
// (a step past the end is not added).
template <int BITS, bool CODEBOOK, int NG>
__global__ void __launch_bounds__(256, 2) k_project_batch(ProjectArgs a) {
    constexpr int KC = 4;  // steps per chunk: one DMA a token
    constexpr int T = 4 * NG, XS = 64 * KC + 16;  // a token's chunk, padded so that four tokens' reads spread over the banks
    __shared__ __attribute__((aligned(16))) float s_x[2][T][XS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = lane >> 2, i = lane & 3;
    const int r0 = blockIdx.x * 16 + wave * 4, t0 = blockIdx.y * T;
    const int steps = a.cols >> 6, row = min(r0 + i, a.rows - 1);
    const bool gate = BITS == 32 && a.gate_row && row == a.rows - 1;
    const uint8_t *row_codes = gate ? (const uint8_t *)a.gate_row : a.codes + (int64_t)row * a.cols * BITS / 8;
    const int64_t row_groups = BITS >= 16 ? 0 : (int64_t)row * (a.cols >> a.group_shift);
    const float *row_scales = a.scales + row_groups, *row_offsets = (a.has_offset ? a.offsets : a.scales) + row_groups;
    // Each wave brings every fourth token's chunk: 256 columns, 1 KiB, one DMA.
    auto stage = [&](int c, int buf) {
#pragma unroll
        for (int u = 0; u < NG; u++) {
            const int t = wave + 4 * u;
            const float *x = a.X + (int64_t)min(t0 + t, a.tokens - 1) * a.cols;
            __builtin_amdgcn_global_load_lds(x + min(64 * KC * c + 4 * lane, a.cols - 4), (lds_void_t *)&s_x[buf][t][0], 16,
                                             0, 0);
        }
    };
    Raw<BITS> cur[KC], next[KC];
    auto load = [&](int c, Raw<BITS> (&w)[KC]) {
#pragma unroll
        for (int k = 0; k < KC; k++)
            load_raw<BITS>(a, row_codes, row_scales, row_offsets, 64 * min(KC * c + k, steps - 1) + 4 * b, w[k]);
    };
    f32x4 acc[NG][4];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[g][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 xv[2][NG];  // the tokens' columns of this step and of the next
    auto read_x = [&](int buf, int k) {
#pragma unroll
        for (int g = 0; g < NG; g++) xv[k & 1][g] = *(const f32x4 *)&s_x[buf][4 * g + i][64 * k + 4 * b];
    };
    auto step = [&](int k, const Raw<BITS> &raw, bool live) {
        float w[4];
        widen<BITS, CODEBOOK>(a, raw, w);
#pragma unroll
        for (int q = 0; q < 4; q++) w[q] = live ? w[q] : 0.0f;
#pragma unroll
        for (int g = 0; g < NG; g++) {
            f32x4 p[4];
#pragma unroll
            for (int q = 0; q < 4; q++)
                p[q] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv[k & 1][g][q], w[q], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; q++) acc[g][q] = acc[g][q] + p[q];
        }
    };
    const int chunks = (steps + KC - 1) / KC, rest = steps - KC * (chunks - 1);  // `rest` steps in the last chunk
    stage(0, 0);
    load(0, cur);
    for (int c = 0; c < chunks; c++) {
        // Chunk c has landed for every wave, and nobody reads the buffer of
        // chunk c - 1 any more.
        __builtin_amdgcn_s_waitcnt(0 | 0x7 << 4 | 0xF << 8);  // vmcnt(0)
        __syncthreads();
        // (the weights' loads run past the end, on the last step: a load under
        // a condition would have to be waited for at once)
        load(c + 1, next);
        if (c + 1 < chunks) {
            stage(c + 1, (c + 1) & 1);
        } else if (rest < KC) {
            // steps past the end: columns and weights of 0, which no partial sum notices
            for (int t = wave; t < T; t += 4)
                for (int col = 64 * rest + lane; col < 64 * KC; col += 64) s_x[c & 1][t][col] = 0.0f;
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < KC; k++) {
            if (k == 0) read_x(c & 1, 0);
            if (k + 1 < KC) read_x(c & 1, k + 1);
            // (one step's products at a time: the accumulators leave no room for more)
            __builtin_amdgcn_sched_barrier(0);
            step(k, cur[k], KC * c + k < steps);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int k = 0; k < KC; k++) cur[k] = next[k];
    }
    const int quarter = lane >> 4, token = quarter == 1 ? 2 : quarter == 2 ? 1 : quarter;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        float y = tree_columns(acc[g]);
        const int t = t0 + 4 * g + token;
        if ((lane & 15) < 4 && r0 + i < a.rows && t < a.tokens) {
            if (gate) {
                a.gate_out[t] = y;
            } else {
                if (BITS == 32 && a.expert_bias) y = y + a.expert_bias[r0 + i];
                a.Y[(int64_t)t * a.stride + a.out + r0 + i] = y;
            }
        }
    }
}

// strata_quant_gemv (kernels/strata.cu:134-155: strata_quant_project's
// arithmetic for one token). The same lanes as above, with the products on
// the vector unit: a wave owns four rows, lane l the columns 4 (l / 4) .. + 3
// of every step for row l % 4. The wave's codes, scales and offsets and the
// block's copy of x all arrive by DMA at once, and the steps run from LDS:
// four weights for a code, a scale, an offset and a 16-byte x read, where one
// weight a lane cost three reads. Code rows lie 2 BITS words apart modulo 32,
// so that the four rows of a step meet different banks. Bound: the vector
// instructions (seven a weight) and the stream about equally. 2,560 x 10,240
// with 32-weight groups and offsets, from a graph, us: 4 bits 13.7 -> 10.4, 8
// bits 20.1 -> 14.6; 3,072 x 300 at 8 bits 11.2 -> 7.7.
//
// PIECES: rows whose LDS leaves a CU few waves come in pieces of 1,024 or 2,048
// columns, the sums going on from one to the next. FINE: groups of one and two
// weights, a scale a column.
constexpr uint64_t kOneTokenLds = 65536;
__host__ __device__ constexpr int one_token_pitch(int bits, int cols) {
    const int words = cols * bits / 32;
    return words + (2 * bits + 32 - words % 32) % 32;
}
// Groups of a row, or those that a piece of it holds or lies in (group sizes are powers of two).
__host__ __device__ constexpr int one_token_groups(int piece, int shift) { return (piece >> shift) > 0 ? piece >> shift : 1; }
enum OneToken { WHOLE, FINE, PIECES };
template <int BITS, bool CODEBOOK, OneToken MODE>
__global__ void __launch_bounds__(256) k_project_one(ProjectArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint32_t s_one[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int b = lane >> 2, i = lane & 3, piece = MODE == PIECES ? a.tokens : a.cols;  // (one token: its slot holds the piece)
    const int row_words = a.cols * BITS / 32, row_groups = a.cols >> a.group_shift;
    const int pitch = one_token_pitch(BITS, piece), ng = MODE == PIECES ? one_token_groups(piece, a.group_shift) : row_groups;
    float *s_x = (float *)s_one;
    uint32_t *codes = s_one + piece + wave * 4 * (pitch + 2 * ng);
    float *scales = (float *)(codes + 4 * pitch), *offsets = scales + 4 * ng;
    const int r0 = (blockIdx.x * waves + wave) * 4, nr = min(4, a.rows - r0);
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int p0 = 0; MODE != PIECES || p0 < a.cols; p0 += piece) {
        const int n = MODE == PIECES ? min(piece, a.cols - p0) : a.cols, words = n * BITS / 32, g0 = p0 >> a.group_shift;
        if (p0) __syncthreads();  // the last piece has been read
        for (int c = 256 * wave; c < n; c += 256 * waves)
            if (c + 4 * lane < n)
                __builtin_amdgcn_global_load_lds(a.X + p0 + c + 4 * lane, (lds_void_t *)(s_x + c), 16, 0, 0);
        for (int r = 0; r < nr; r++) {
            const uint8_t *src = a.codes + ((int64_t)(r0 + r) * row_words + p0 * BITS / 32) * 4;
            for (int c = 0; c < words; c += 256)
                if (c + 4 * lane < words)
                    __builtin_amdgcn_global_load_lds(src + 4 * (c + 4 * lane), (lds_void_t *)(codes + r * pitch + c), 16, 0, 0);
        }
        // (four rows' groups are whole 16-byte pieces, fewer rows' may not be;
        // PIECES: one row's are if they are in every piece)
        auto groups = [&](const float *src, float *dst) {
            src += (int64_t)r0 * row_groups;
            if constexpr (MODE == PIECES) {
                const int ngp = ((p0 + n - 1) >> a.group_shift) - g0 + 1;
                for (int r = 0; r < nr; r++) {
                    const float *from = src + (int64_t)r * row_groups + g0;
                    float *to = dst + r * ng;
                    if (((row_groups | g0 | ngp | ng) & 3) == 0) {
                        for (int c = 0; c < ngp; c += 256)
                            if (c + 4 * lane < ngp)
                                __builtin_amdgcn_global_load_lds(from + c + 4 * lane, (lds_void_t *)(to + c), 16, 0, 0);
                    } else {
                        for (int c = 0; c < ngp; c += 64)
                            if (c + lane < ngp) __builtin_amdgcn_global_load_lds(from + c + lane, (lds_void_t *)(to + c), 4, 0, 0);
                    }
                }
            } else if (nr == 4) {
                for (int c = 0; c < 4 * ng; c += 256)
                    if (c + 4 * lane < 4 * ng)
                        __builtin_amdgcn_global_load_lds(src + c + 4 * lane, (lds_void_t *)(dst + c), 16, 0, 0);
            } else {
                for (int c = 0; c < nr * ng; c += 64)
                    if (c + lane < nr * ng) __builtin_amdgcn_global_load_lds(src + c + lane, (lds_void_t *)(dst + c), 4, 0, 0);
            }
        };
        groups(a.scales, scales);
        if (a.has_offset) groups(a.offsets, offsets);
        __builtin_amdgcn_s_waitcnt(0 | 0x7 << 4 | 0xF << 8);  // vmcnt(0)
        __syncthreads();
        if (nr < 1) {
            if (MODE == PIECES) continue;
            return;
        }
        const int row = min(i, nr - 1), steps = n >> 6;
        const uint8_t *code = (const uint8_t *)(codes + row * pitch) + b * BITS / 2;
        const float *sc = scales + row * ng, *of = (a.has_offset ? offsets : scales) + row * ng, *x = s_x + 4 * b;
        constexpr int UNROLL = MODE == FINE ? 4 : 8;
#pragma unroll UNROLL
        for (int k = 0; k < steps; k++) {
            Raw<BITS> raw;
            const uint8_t *c = code + k * 8 * BITS;
            raw.code[0] = BITS == 8 ? *(const uint32_t *)c : BITS == 4 ? *(const uint16_t *)c : *c;
            const int col = p0 + 64 * k + 4 * b, g = (col >> a.group_shift) - g0;
            const f32x4 xv = *(const f32x4 *)(x + 64 * k);
            float w[4];
            if constexpr (MODE == FINE) {
                unpack<BITS, CODEBOOK>(a, raw.code[0], w);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int gq = (col + q) >> a.group_shift;
                    w[q] = w[q] * sc[gq];
                    w[q] = w[q] + (a.has_offset ? of[gq] : 0.0f);
                }
            } else {
                raw.scale = sc[g];
                raw.offset = of[g];
                widen<BITS, CODEBOOK>(a, raw, w);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) sum[q] = sum[q] + w[q] * xv[q];
        }
        if constexpr (MODE != PIECES) break;
    }
    if (MODE == PIECES && nr < 1) return;
    // the reference's tree: columns 32, 16, 8 and 4 apart are lanes, 2 and 1 are q
#pragma unroll
    for (int q = 0; q < 4; q++) {
        float v = sum[q];
        v = v + __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false)[1]);
        v = v + __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false)[1]);
        v = v + sm::dpp_f32<0x108>(0.0f, v);
        sum[q] = v + sm::dpp_f32<0x104>(0.0f, v);
    }
    if (lane < nr) a.Y[r0 + lane] = (sum[0] + sum[2]) + (sum[1] + sum[3]);
}

template <int BITS, bool CODEBOOK>
void launch(sm_ctx *ctx, const ProjectArgs &a, int ng) {
    const dim3 grid((unsigned)((a.rows + 15) / 16), (unsigned)((a.tokens + 4 * ng - 1) / (4 * ng)));
    switch (ng) {
        case 1: k_project_batch<BITS, CODEBOOK, 1><<<grid, 256, 0, ctx->stream>>>(a); break;
        case 2: k_project_batch<BITS, CODEBOOK, 2><<<grid, 256, 0, ctx->stream>>>(a); break;
        default: k_project_batch<BITS, CODEBOOK, 4><<<grid, 256, 0, ctx->stream>>>(a); break;
    }
}

// Groups of tokens per wave. More of them share a weight's load and
// widening, fewer make more blocks. Measured at 2,560 columns, a block
// takes 8 / 10 / 17 us (1 / 2 / 4 groups) where every CU has one, and
// 5 / 5 / 7 us for each further one a CU has to take; the least of those
// sums is taken. bf16, in us with 1 / 2 / 4 groups: 10,240 rows x 4
// tokens 17 / 20 / 31, x 16 54 / 31 / 31, x 32 105 / 58 / 49; 2,560 rows
// x 12 12 / 14 / 17, x 16 18 / 14 / 17, x 32 28 / 20 / 23; 600 rows x 16
// 10.5 / 10.7 / 17.
int token_groups(int rows, int tokens) {
    const int first[3] = {8, 10, 17}, further[3] = {5, 5, 7};
    int ng = 1, best = 0;
    for (int k = 0; k < 3; k++) {
        const int64_t blocks = (int64_t)((rows + 15) / 16) * ((tokens + (4 << k) - 1) / (4 << k));
        const int cost = first[k] + further[k] * (int)std::min<int64_t>((blocks - 1) / 256, 1 << 20);
        if (k == 0 || cost < best) {
            ng = 1 << k;
            best = cost;
        }
    }
    return ng;
}

}  // namespace

namespace smi {

// Fewer outputs leave the batch kernel's blocks to a chain of load latencies,
// which the general kernels' wave per output beats. Measured from graphs, three
// matrices in turn, general over batch: bf16, 64 to 12,288 columns and 2 to 64
// tokens, 0.62 to 0.99 at 2,600 outputs, 0.65 to 1.02 at 3,000, 0.81 to 1.13 at
// 3,800, 0.92 to 1.25 at 4,200 and 1.02 to 1.42 at 5,400. The quantized general
// kernels do more per weight: 1.00 to 1.66 at 2,600 to 2,900 outputs (fewer
// were not measured over these ranges).
int64_t batch_min_outputs(int bits) { return bits == 16 ? 4096 : 2560; }

bool project_batch_takes(int bits, int cols, int rows, int tokens, uint64_t X, uint64_t codes, int group, int bias,
                         int codebook) {
    if (tokens < 2 || (int64_t)rows * tokens < batch_min_outputs(bits) || cols % 64 || X % 16 || codes % 8) return false;
    if (bits == 16) return true;
    if (group < 4 || (group & (group - 1)) || (codebook == 1 && bits != 4)) return false;
    return bias > -(1 << 23) && bias < (1 << 23) - 256;
}

int project_batch(sm_ctx *ctx, int bits, const float *X, const void *codes, const float *scales, const float *offsets,
                  float *Y, int cols, int rows, int tokens, int stride, int out, int group, int bias, int codebook,
                  int has_offset) {
    ProjectArgs a = {X, (const uint8_t *)codes, scales, offsets, Y, cols, rows, tokens, stride, out, 0, has_offset, (float)bias, nullptr, nullptr, nullptr};
    while (bits != 16 && (1 << a.group_shift) < group) a.group_shift++;
    const int ng = token_groups(rows, tokens);
    switch (bits) {
        case 2: launch<2, false>(ctx, a, ng); break;
        case 4: codebook == 1 ? launch<4, true>(ctx, a, ng) : launch<4, false>(ctx, a, ng); break;
        case 8: launch<8, false>(ctx, a, ng); break;
        default: launch<16, false>(ctx, a, ng); break;
    }
    return launched(ctx);
}

bool route_batch_takes(const float *X, int width, const float *Wr, const float *gate_w) {
    return width % 64 == 0 && ((uintptr_t)X | (uintptr_t)Wr | (uintptr_t)gate_w) % 16 == 0;
}

int route_batch(sm_ctx *ctx, const float *X, int tokens, int width, const float *Wr, const float *bias, int experts,
                float *logits, const float *gate_w, float *gate_out) {
    const ProjectArgs a = {X, (const uint8_t *)Wr, nullptr, nullptr, logits, width, experts + (gate_w ? 1 : 0), tokens, experts, 0,
                           0, 0, 0.0f, gate_w, bias, gate_out};
    launch<32, false>(ctx, a, token_groups(a.rows, tokens));
    return launched(ctx);
}

static int log2_of(int n) { return 31 - __builtin_clz((unsigned)n); }
// LDS of a block of `waves` waves and pieces of `piece` columns; the most
// waves that kOneTokenLds holds, and how many of them a CU does.
static uint64_t one_token_lds(int bits, int piece, int shift, int waves) {
    return 4ull * (piece + (uint64_t)waves * 4 * (one_token_pitch(bits, piece) + 2 * one_token_groups(piece, shift)));
}
static int one_token_waves(int bits, int piece, int shift) {
    int waves = 4;
    while (waves > 0 && one_token_lds(bits, piece, shift, waves) > kOneTokenLds) waves--;
    return waves;
}
static int one_token_waves_per_cu(int bits, int piece, int shift) {
    const int waves = one_token_waves(bits, piece, shift);
    return waves ? waves * (int)(163840 / one_token_lds(bits, piece, shift, waves)) : 0;
}

bool project_one_takes(int bits, int cols, int rows, uint64_t X, uint64_t codes, uint64_t scales, uint64_t offsets, int group,
                       int bias, int codebook) {
    if (cols % 64 || (X | codes | scales | offsets) % 16) return false;
    if ((group & (group - 1)) || (codebook == 1 && bits != 4)) return false;
    // Groups of one and two weights, whose scales are most of a row: up to 256
    // a row, and only with many rows (8 bits, general over this: 256 columns in
    // groups of one 3.8 / 4.5 us at 300 rows, 4.8 / 4.6 at 3,072, 9.2 / 7.7 at
    // 10,240).
    if (group < 4 && (cols / group > 256 || rows <= 2048)) return false;
    return bias > -(1 << 23) && bias < (1 << 23) - 256 && one_token_waves(bits, cols, log2_of(group)) > 0;
}

template <OneToken MODE>
static auto one_token_kernel(int bits, int codebook) {
    return bits == 2   ? k_project_one<2, false, MODE>
           : bits == 8 ? k_project_one<8, false, MODE>
                       : (codebook == 1 ? k_project_one<4, true, MODE> : k_project_one<4, false, MODE>);
}

int project_one(sm_ctx *ctx, int bits, const float *X, const void *codes, const float *scales, const float *offsets, float *Y,
                int cols, int rows, int group, int bias, int codebook, int has_offset) {
    // Pieces once whole rows leave a CU six waves or fewer, the rows fill the
    // GPU more than once and pieces at least double the waves; the shorter ones
    // where the longer leave fewer than twelve and more than one round. 10,240
    // rows of 8 bits, whole / in pieces, us: 4,096 columns 35.8 / 20.6 with
    // 16-weight groups (27.7 in the longer ones) and 26.8 / 19.4 with 32; 6,144
    // columns 55.6 / 24.0; 2,100 rows of 4,096 9.3 / 9.6.
    const int shift = log2_of(group), whole = one_token_waves_per_cu(bits, cols, shift);
    int piece = cols;
    if (cols >= 4096 && whole <= 6 && rows > 256 * 4 * whole)
        for (int p : {2048, 1024}) {
            const int per_cu = one_token_waves_per_cu(bits, p, shift);
            if (per_cu >= 2 * whole) piece = p;
            if (per_cu >= 12 || rows <= 256 * 4 * per_cu) break;
        }
    const bool pieces = piece < cols;
    const int waves = one_token_waves(bits, piece, shift);
    const ProjectArgs a = {X,  (const uint8_t *)codes, scales, offsets,    Y,          cols,    rows,    pieces ? piece : 1,
                           rows, 0, shift, has_offset, (float)bias, nullptr, nullptr, nullptr};
    const auto k = pieces      ? one_token_kernel<PIECES>(bits, codebook)
                   : group < 4 ? one_token_kernel<FINE>(bits, codebook)
                               : one_token_kernel<WHOLE>(bits, codebook);
    k<<<(unsigned)((rows + 4 * waves - 1) / (4 * waves)), 64 * waves, one_token_lds(bits, piece, shift, waves), ctx->stream>>>(a);
    return launched(ctx);
}

}  // namespace smi
