// The shrink to Q2_K: super-blocks of Q3_K, Q4_K or Q5_K re-encoded as Q2_K on the GPU, plain or
// with per-column importance weights.
//
// Restates crates/engine/src/requant.rs:113-304 (fit16, q2k_encode, q2k_encode_w and the six
// coachwhip_requant_* kernels). The reference runs one thread per 256-weight super-block with
// all 256 values in its registers; here 16 lanes share a super-block, lane j holding sub-block j
// (values 16j..16j+15), which is the unit fit16 works on:
//  1. each lane dequantizes its 16 values (candle's to_float arithmetic: a small integer times
//     an f32 product of f16 fields, minus another; the shader's dq_* readers give the same
//     values) and takes their min and max;
//  2. it runs fit16 (two weighted least-squares rounds) on its own;
//  3. the block's largest scale and min come from a butterfly over the 16 lanes, each lane
//     putting its scale and min on the 4-bit grid and rounding its 16 quants;
//  4. lane j's quants land in bytes 32(j/8) + 16(j%2) + i at bit 2((j%8)/2): the four lanes that
//     share those 16 bytes OR their words together through two shuffles, and one of them stores.
// Arithmetic is IEEE f32 in the shader's order, with no contraction into FMAs and correctly
// rounded division and square root, so the output bytes equal a CPU restatement's exactly. The
// 48 divisions per lane whose quotients only pick one of four levels are replaced by comparisons of
// the numerator with the exact places where the rounded result steps (Steps); sums that do not
// change between the fit's rounds are taken once, and the plain shrink has no weights to multiply.
// VALU-bound: 32 experts of config 5's shape (Q3_K gate and up, Q5_K down, 85 MB in and out) in
// three launches, 215 -> 109 us (weighted 250 -> 156); about 960 VALU instructions per lane, 2,100 before.
#include "cw_common.h"
#include "cw_requant.h"

namespace cw {
namespace {

__device__ __forceinline__ float max_sel(float a, float b) { return b > a ? b : a; }
// min(15, (int)v) with a saturating conversion (NaN gives 0)
__device__ __forceinline__ int level15(float v) { return v >= 15.f ? 15 : v >= 1.f ? (int)v : 0; }

__device__ __forceinline__ float f16_at(const uint8_t *p) {
    uint16_t h;
    __builtin_memcpy(&h, p, 2);
    return (float)__builtin_bit_cast(_Float16, h);
}

// sub-block j of 6-bit scale / min pairs packed in 12 bytes (vendor/candle-core/src/quantized/utils.rs:50-60)
__device__ __forceinline__ void scale_min_k4(int j, const uint8_t *q, int &d, int &m) {
    if (j < 4) {
        d = q[j] & 63;
        m = q[j + 4] & 63;
    } else {
        d = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// The level of n: clamp((int)(n / scale + 0.5f), 0, 3), quotient and sum rounded to f32 (0 for a NaN, and
// for a scale that is not above 0). Both roundings are monotone, so level >= k means n > scale M_k, with
// M_k the midpoint below the smallest quotient whose sum reaches k: that quotient is 0.5 - 2^-25 for k = 1
// (whose sum 1 - 2^-25 ties to 1), and 1.5 and 2.5. n / scale cannot equal M_k: an odd multiple of 25
// significant bits times scale needs more than n's 24. scale M_k has 49 bits, exact in f64; step k is the
// smallest f32 above it. A product past f32 gives +inf (reached by n = inf alone), an infinite scale a NaN
// (never reached, as inf / inf is no level).
struct Steps {
    float t1, t2, t3;
    static __device__ __forceinline__ float above(double v) {
        const float f = (float)v;
        return (double)f <= v ? __uint_as_float(__float_as_uint(f) + 1u) : f;
    }
    __device__ __forceinline__ Steps(float scale) {
        const double s = (double)scale;
        const bool on = scale > 0.f;
        const float never = __uint_as_float(0x7fc00000u);
        t1 = on ? above(s * (0.5 - 0x1.8p-25)) : never;
        t2 = on ? above(s * (1.5 - 0x1p-24)) : never;
        t3 = on ? above(s * (2.5 - 0x1p-23)) : never;
    }
    __device__ __forceinline__ float level(float n) const { return n >= t3 ? 3.f : n >= t2 ? 2.f : n >= t1 ? 1.f : 0.f; }
    __device__ __forceinline__ uint32_t ilevel(float n) const { return n >= t3 ? 3u : n >= t2 ? 2u : n >= t1 ? 1u : 0u; }
};

// x[i] = value 16 g + i of a source super-block b (g = the lane's sub-block), four codes per dword
template <int SRC>
__device__ __forceinline__ void dequant16(const uint8_t *b, int g, float *x);
__device__ __forceinline__ uint4 load16(const uint8_t *p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
__device__ __forceinline__ float code(uint32_t w, int i) { return (float)((w >> (8 * i)) & 0xFFu); }

// Q3_K {hmask[32], qs[64], scales[12], d}: k_quants.rs:1514-1571 (a clear hmask bit takes 4 off the code)
template <>
__device__ __forceinline__ void dequant16<CW_Q3_K>(const uint8_t *b, int g, float *x) {
#pragma clang fp contract(off)
    const int half = g >> 3, ss = (g >> 1) & 3, part = g & 1;
    const int lo = (b[96 + (g & 7)] >> (4 * (g >> 3))) & 0xF, hi = (b[104 + (g & 3)] >> (2 * (g >> 2))) & 3;
    const float dl = f16_at(b + 108) * ((float)(lo | (hi << 4)) - 32.0f);
    const uint4 q = load16(b + 32 + 32 * half + 16 * part), h = load16(b + 16 * part);
    const int hs = 4 * half + ss;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t c = (((&q.x)[k] >> (2 * ss)) & 0x03030303u) | ((((&h.x)[k] >> hs) & 0x01010101u) << 2);
#pragma unroll
        for (int i = 0; i < 4; i++) x[4 * k + i] = dl * (code(c, i) - 4.0f);
    }
}

// Q4_K {d, dmin, scales[12], qs[128]}: k_quants.rs:1821-1849
template <>
__device__ __forceinline__ void dequant16<CW_Q4_K>(const uint8_t *b, int g, float *x) {
#pragma clang fp contract(off)
    const int c4 = g >> 2, upper = (g >> 1) & 1;
    int s, m;
    scale_min_k4(2 * c4 + upper, b + 4, s, m);
    const float d1 = f16_at(b) * (float)s, m1 = f16_at(b + 2) * (float)m;
    const uint4 q = load16(b + 16 + 32 * c4 + 16 * (g & 1));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t c = ((&q.x)[k] >> (4 * upper)) & 0x0F0F0F0Fu;
#pragma unroll
        for (int i = 0; i < 4; i++) x[4 * k + i] = d1 * code(c, i) - m1;
    }
}

// Q5_K {d, dmin, scales[12], qh[32], qs[128]}: k_quants.rs:2120-2152
template <>
__device__ __forceinline__ void dequant16<CW_Q5_K>(const uint8_t *b, int g, float *x) {
#pragma clang fp contract(off)
    const int c4 = g >> 2, upper = (g >> 1) & 1;
    int s, m;
    scale_min_k4(2 * c4 + upper, b + 4, s, m);
    const float d1 = f16_at(b) * (float)s, m1 = f16_at(b + 2) * (float)m;
    const uint4 q = load16(b + 48 + 32 * c4 + 16 * (g & 1)), h = load16(b + 16 + 16 * (g & 1));
    const int hb = 2 * c4 + upper;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t c = (((&q.x)[k] >> (4 * upper)) & 0x0F0F0F0Fu) | ((((&h.x)[k] >> hb) & 0x01010101u) << 4);
#pragma unroll
        for (int i = 0; i < 4; i++) x[4 * k + i] = d1 * code(c, i) - m1;
    }
}

// fit16, requant.rs:119-138. Plain (W false): every weight is 1, and products with it are the other
// factor. The sums of w and of w x are the same in both rounds.
template <bool W>
__device__ __forceinline__ void fit16(const float *x, const float *w, float &scale, float &mn) {
#pragma clang fp contract(off)
    float sw = 0.f, swx = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        sw += W ? w[i] : 1.f;
        swx += W ? w[i] * x[i] : x[i];
    }
#pragma unroll
    for (int round = 0; round < 2; ++round) {
        float swl = 0.f, swll = 0.f, swlx = 0.f;
        const Steps st(scale);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float fl = st.level(x[i] + mn), wl = W ? w[i] * fl : fl;
            swl += wl;
            swll += wl * fl;
            swlx += wl * x[i];
        }
        const float det = sw * swll - swl * swl;
        if (det > 1e-12f) {
            const float a = (sw * swlx - swl * swx) / det;
            const float b = (swl * swlx - swll * swx) / det;
            if (a > 0.f && b >= 0.f) {
                scale = a;
                mn = b;
            }
        }
    }
}

// One super-block per 16 lanes (g = lane % 16 = this lane's sub-block): src is the source block,
// w_row the block's 256 column weights (W), y the 84-byte Q2_K block (stored when store is set;
// every lane takes part in the shuffles either way).
template <int SRC, bool W>
__device__ __forceinline__ void shrink_block(const uint8_t *src, const float *w_row, uint8_t *y, int g, bool store) {
#pragma clang fp contract(off)
    float x[16], w[16];
    dequant16<SRC>(src, g, x);
    if constexpr (W) {
        const float *ws = w_row + 16 * g;
#pragma unroll
        for (int i = 0; i < 16; i++) w[i] = sqrtf(max_sel(ws[i], 0.f)) + 1e-6f;
    }
    // the shader's running selects (b < a ? b : a) keep a NaN in x[0] and pass over later ones, as a
    // minimum that prefers numbers does from a numeric x[0] (zeros' signs do not reach the output)
    float lo = x[0], hi = x[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) {
        lo = fminf(lo, x[i]);
        hi = fmaxf(hi, x[i]);
    }
    if (x[0] != x[0]) lo = hi = x[0];
    if (lo > 0.f) lo = 0.f;
    float sc = (hi - lo) / 3.f, mn = -lo;
    fit16<W>(x, w, sc, mn);
    // the block's maxima, started from +0 as the shader's running maximum is
    float max_scale = max_sel(0.f, sc), max_min = max_sel(0.f, mn);
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) {
        max_scale = max_sel(max_scale, __shfl_xor(max_scale, o, 64));
        max_min = max_sel(max_min, __shfl_xor(max_min, o, 64));
    }
    const float inv_scale = max_scale > 0.f ? 15.f / max_scale : 0.f;
    const float inv_min = max_min > 0.f ? 15.f / max_min : 0.f;
    const int ls = level15(sc * inv_scale + 0.5f), lm = level15(mn * inv_min + 0.5f);
    const _Float16 dh = (_Float16)(max_scale / 15.f), mh = (_Float16)(max_min / 15.f);
    const float dj = (float)dh * (float)ls, mj = (float)mh * (float)lm;
    const int shift = 2 * ((g >> 1) & 3);
    uint32_t word[4] = {0u, 0u, 0u, 0u};
    const Steps st(dj);
#pragma unroll
    for (int i = 0; i < 16; ++i) word[i >> 2] |= st.ilevel(x[i] + mj) << (8 * (i & 3));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        word[k] <<= shift;
        word[k] |= (uint32_t)__shfl_xor((int)word[k], 2, 64);
        word[k] |= (uint32_t)__shfl_xor((int)word[k], 4, 64);
    }
    if (!store) return;
    y[g] = (uint8_t)(ls | (lm << 4));
    if (shift == 0) {
        uint8_t *qs = y + 16 + 32 * (g >> 3) + 16 * (g & 1);
#pragma unroll
        for (int k = 0; k < 4; k++) __builtin_memcpy(qs + 4 * k, &word[k], 4);
    }
    if (g == 0) {
        const uint32_t dd = (uint32_t)__builtin_bit_cast(uint16_t, dh) | ((uint32_t)__builtin_bit_cast(uint16_t, mh) << 16);
        __builtin_memcpy(y + 80, &dd, 4);
    }
}

template <int SRC>
constexpr int src_bytes() { return SRC == CW_Q3_K ? 110 : SRC == CW_Q4_K ? 144 : 176; }

// n_blocks consecutive source blocks into n_blocks consecutive Q2_K blocks
template <int SRC, bool W>
__global__ __launch_bounds__(256) void k_requant_q2k(const uint8_t *src, int64_t n_blocks, const float *shape,
                                                     int64_t blocks_per_row, uint8_t *dst) {
    const int g = threadIdx.x & 15;
    const int64_t blk = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    // every lane joins the shuffles; lanes past the end work on the last block and store nothing
    const int64_t b = blk < n_blocks ? blk : n_blocks - 1;
    shrink_block<SRC, W>(src + b * src_bytes<SRC>(), W ? shape + (b % blocks_per_row) * 256 : nullptr, dst + b * 84, g, blk < n_blocks);
}

// Piece y (blockIdx.y) of a list: blocks_per_piece source blocks at src + y * src_stride into
// dst + index[y] * dst_stride (the bank's shrink of staged experts into their slots)
template <int SRC, bool W>
__global__ __launch_bounds__(256) void k_shrink_pieces(const uint8_t *src, int64_t src_stride, ShrinkIndex index, uint8_t *dst,
                                                       int64_t dst_stride, int64_t blocks_per_piece, const float *shape,
                                                       int64_t blocks_per_row) {
    const int g = threadIdx.x & 15;
    const int64_t blk = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    const int64_t b = blk < blocks_per_piece ? blk : blocks_per_piece - 1;
    const uint8_t *s = src + blockIdx.y * src_stride + b * src_bytes<SRC>();
    uint8_t *y = dst + (int64_t)index.i[blockIdx.y] * dst_stride + b * 84;
    shrink_block<SRC, W>(s, W ? shape + (b % blocks_per_row) * 256 : nullptr, y, g, blk < blocks_per_piece);
}

}  // namespace

int shrink_pieces(int src_dtype, const uint8_t *src, int64_t src_stride, const ShrinkIndex &index, int n, uint8_t *dst,
                  int64_t dst_stride, int64_t blocks_per_piece, const float *shape, int64_t blocks_per_row, hipStream_t s) {
    if (n == 0 || blocks_per_piece == 0) return CW_OK;
    const dim3 grid((unsigned)((blocks_per_piece + 15) / 16), (unsigned)n), block(256);
    switch (src_dtype) {
    case CW_Q3_K:
        if (shape) hipLaunchKernelGGL((k_shrink_pieces<CW_Q3_K, true>), grid, block, 0, s, src, src_stride, index, dst, dst_stride, blocks_per_piece, shape, blocks_per_row);
        else hipLaunchKernelGGL((k_shrink_pieces<CW_Q3_K, false>), grid, block, 0, s, src, src_stride, index, dst, dst_stride, blocks_per_piece, shape, blocks_per_row);
        break;
    case CW_Q4_K:
        if (shape) hipLaunchKernelGGL((k_shrink_pieces<CW_Q4_K, true>), grid, block, 0, s, src, src_stride, index, dst, dst_stride, blocks_per_piece, shape, blocks_per_row);
        else hipLaunchKernelGGL((k_shrink_pieces<CW_Q4_K, false>), grid, block, 0, s, src, src_stride, index, dst, dst_stride, blocks_per_piece, shape, blocks_per_row);
        break;
    case CW_Q5_K:
        if (shape) hipLaunchKernelGGL((k_shrink_pieces<CW_Q5_K, true>), grid, block, 0, s, src, src_stride, index, dst, dst_stride, blocks_per_piece, shape, blocks_per_row);
        else hipLaunchKernelGGL((k_shrink_pieces<CW_Q5_K, false>), grid, block, 0, s, src, src_stride, index, dst, dst_stride, blocks_per_piece, shape, blocks_per_row);
        break;
    default: return set_error(CW_ENOTSUP, "shrink: source type %d (Q3_K, Q4_K or Q5_K)", src_dtype);
    }
    return check_launch("k_shrink_pieces");
}

static int requant_q2k(int src_dtype, const void *src, int64_t n_blocks, const float *shape, int64_t blocks_per_row,
                       void *dst, hipStream_t s) {
    if (n_blocks == 0) return CW_OK;
    const dim3 grid((unsigned)((n_blocks + 15) / 16)), block(256);
    const uint8_t *in = (const uint8_t *)src;
    uint8_t *out = (uint8_t *)dst;
    switch (src_dtype) {
    case CW_Q3_K:
        if (shape) hipLaunchKernelGGL((k_requant_q2k<CW_Q3_K, true>), grid, block, 0, s, in, n_blocks, shape, blocks_per_row, out);
        else hipLaunchKernelGGL((k_requant_q2k<CW_Q3_K, false>), grid, block, 0, s, in, n_blocks, shape, blocks_per_row, out);
        break;
    case CW_Q4_K:
        if (shape) hipLaunchKernelGGL((k_requant_q2k<CW_Q4_K, true>), grid, block, 0, s, in, n_blocks, shape, blocks_per_row, out);
        else hipLaunchKernelGGL((k_requant_q2k<CW_Q4_K, false>), grid, block, 0, s, in, n_blocks, shape, blocks_per_row, out);
        break;
    case CW_Q5_K:
        if (shape) hipLaunchKernelGGL((k_requant_q2k<CW_Q5_K, true>), grid, block, 0, s, in, n_blocks, shape, blocks_per_row, out);
        else hipLaunchKernelGGL((k_requant_q2k<CW_Q5_K, false>), grid, block, 0, s, in, n_blocks, shape, blocks_per_row, out);
        break;
    default: return set_error(CW_ENOTSUP, "requant: source type %d (Q3_K, Q4_K or Q5_K)", src_dtype);
    }
    return check_launch("k_requant_q2k");
}

}  // namespace cw

extern "C" int cw_requant_q2k(int src_dtype, const void *src, int64_t n_blocks, const float *shape,
                              int64_t blocks_per_row, void *dst, cw_stream_t stream) {
    CW_REQUIRE(n_blocks >= 0 && n_blocks < ((int64_t)1 << 35), "requant: %lld blocks", (long long)n_blocks);
    CW_REQUIRE(n_blocks == 0 || (src && dst), "requant: null pointer");
    CW_REQUIRE(!shape || (blocks_per_row > 0 && ((uintptr_t)shape & 3u) == 0),
               "requant: weights need blocks_per_row > 0 (got %lld) and 4-byte alignment", (long long)blocks_per_row);
    return cw::requant_q2k(src_dtype, src, n_blocks, shape, blocks_per_row, dst, (hipStream_t)stream);
}
