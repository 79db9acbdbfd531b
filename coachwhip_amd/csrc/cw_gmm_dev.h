// Device pieces shared by the grouped GEMMs (cw_mfma.hip, cw_mfma_split.hip): fp16 code helpers, the
// formats' fragment decodes, weight windows in LDS and direct global-to-LDS loads.
#pragma once
#include <type_traits>

#include "cw_device.h"
#include "cw_mfma.h"

namespace cw {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pk_mul_u(uint32_t v, uint32_t sc2) {
    f16x2 a = __builtin_bit_cast(f16x2, v), b = __builtin_bit_cast(f16x2, sc2);
    return __builtin_bit_cast(uint32_t, a * b);
}
__device__ __forceinline__ uint4 scale4(uint4 v, uint32_t sc2) {
    return make_uint4(pk_mul_u(v.x, sc2), pk_mul_u(v.y, sc2), pk_mul_u(v.z, sc2), pk_mul_u(v.w, sc2));
}
// Signs of 8 fp16 codes (dword i holds weights 2i, 2i+1; sign bits clear): bit j of b negates
// weight j. With y = b | b << 15, y << (15 - 2i) has bit 2i of b at bit 15 and bit 2i+1 at bit
// 31; a bit-field insert takes exactly those two bits (bits 8 and up of b never reach them).
__device__ __forceinline__ uint32_t bfi_sign(uint32_t s, uint32_t g) { return (s & 0x80008000u) | (g & 0x7FFF7FFFu); }
__device__ __forceinline__ uint4 apply_signs(uint4 g, uint32_t b) {
    // an opaque b keeps the shifts as shifts: with b known to be small the compiler turns
    // (b | b << 15) << c into one quarter-rate 32-bit multiply per dword
    asm("" : "+v"(b));
    const uint32_t y = b | (b << 15);
    return make_uint4(bfi_sign(y << 15, g.x), bfi_sign(y << 13, g.y), bfi_sign(y << 11, g.z), bfi_sign(y << 9, g.w));
}
// fp16 pair of a small integer multiplier (exact below 2048)
__device__ __forceinline__ uint32_t splat_mult(uint32_t v) {
    const float m = (float)v;
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(m, m));
}

// ------------------------------------------------------------------------------ code tables
// Lattice entries as fp16 integers, built at compile time; a kernel copies the one its format
// needs into LDS. Signs are applied arithmetically (apply_signs), not through a table: a random
// 16-byte LDS lookup costs about as much LDS time as two conflict-free ones.
struct U4 { uint32_t x, y, z, w; };
template <int N> struct Tab { U4 v[N]; };

constexpr uint32_t f16_int(uint32_t v) {  // fp16 bits of a small non-negative integer (< 2048)
    if (v == 0) return 0;
    int e = 0;
    for (uint32_t t = v; t >= 2; t >>= 1) e++;
    return (uint32_t)((e + 15) << 10) | ((v << (10 - e)) & 0x3FFu);
}
constexpr U4 pack8(uint64_t bytes) {
    uint32_t h[8] = {};
    for (int b = 0; b < 8; b++) h[b] = f16_int((uint32_t)(bytes >> (8 * b)) & 0xFF);
    return U4{h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16};
}
constexpr Tab<256> make_iq2xxs_f16() {
    constexpr uint64_t g[256] = {CW_IQ2XXS_GRID_VALUES};
    Tab<256> t{};
    for (int i = 0; i < 256; i++) t.v[i] = pack8(g[i]);
    return t;
}
constexpr Tab<1024> make_iq2s_f16() {
    constexpr uint64_t g[1024] = {CW_IQ2S_GRID_VALUES};
    Tab<1024> t{};
    for (int i = 0; i < 1024; i++) t.v[i] = pack8(g[i]);
    return t;
}
constexpr Tab<256> make_iq3s_f16() {  // two 4-value entries per U4: entry 2i in x,y and 2i+1 in z,w
    constexpr uint32_t g[512] = {CW_IQ3S_GRID_VALUES};
    Tab<256> t{};
    for (int i = 0; i < 256; i++) {
        const U4 a = pack8((uint64_t)g[2 * i] | ((uint64_t)g[2 * i + 1] << 32));
        t.v[i] = a;
    }
    return t;
}
constexpr Tab<128> make_iq3xxs_f16() {  // two 4-value entries per U4: entry 2i in x,y and 2i+1 in z,w
    constexpr uint32_t g[256] = {CW_IQ3XXS_GRID_VALUES};
    Tab<128> t{};
    for (int i = 0; i < 128; i++) t.v[i] = pack8((uint64_t)g[2 * i] | ((uint64_t)g[2 * i + 1] << 32));
    return t;
}
static __constant__ Tab<256> c_iq2xxs_f16 = make_iq2xxs_f16();
static __constant__ Tab<1024> c_iq2s_f16 = make_iq2s_f16();
static __constant__ Tab<256> c_iq3s_f16 = make_iq3s_f16();
static __constant__ Tab<128> c_iq3xxs_f16 = make_iq3xxs_f16();

template <int N>
__device__ __forceinline__ void copy_tab(uint8_t *lds, const Tab<N> &t, int tid, int nt) {
    uint4 *d = (uint4 *)lds;
    const uint4 *src = (const uint4 *)&t;
    for (int i = tid; i < N; i += nt) d[i] = src[i];
}

// ------------------------------------------------------------------------------ formats
// Per format: TS bytes per block, SBK weights per scale unit, LDS table bytes, and the decode of
// one K-step (32 weights) of a row from the row's stage window in LDS (the bytes of 8 K-steps:
// one IQ super-block, or 8 MXFP4 blocks): lane group grp takes weights 8*grp..8*grp+7 of the
// step, as 8 fp16 integer codes times a per-lane multiplier.

__device__ __forceinline__ uint32_t lds_u8(const uint8_t *p) { return *p; }
__device__ __forceinline__ uint32_t lds_u16(const uint8_t *p) { uint16_t v; __builtin_memcpy(&v, p, 2); return v; }
__device__ __forceinline__ uint32_t lds_u32(const uint8_t *p) { uint32_t v; __builtin_memcpy(&v, p, 4); return v; }
// 8 bytes at any LDS address: three aligned dwords and a byte shift (a misaligned ds_read_b64
// measured ~2x slower for the whole stage)
__device__ __forceinline__ uint2 lds_u64(const uint8_t *p) {
    const uint32_t a = (uint32_t)(uintptr_t)p & 3;
    const uint32_t *q = (const uint32_t *)(p - a);
    const uint32_t d0 = q[0], d1 = q[1], d2 = q[2];
    return make_uint2(__builtin_amdgcn_alignbyte(d1, d0, a), __builtin_amdgcn_alignbyte(d2, d1, a));
}

// A row's stage window in LDS, with the dword address and byte shift of its 8-byte reads
// (which start ORG bytes into the window) worked out once per stage instead of per read
struct WinRef {
    const uint8_t *p;     // the window: the row's bytes of this stage
    const uint32_t *qa;   // p + ORG rounded down to a dword
    uint32_t sh;          // (p + ORG) & 3
    template <int ORG>
    static __device__ __forceinline__ WinRef at(const uint8_t *p) {
        const uint32_t o = (uint32_t)(uintptr_t)(p + ORG);
        return WinRef{p, (const uint32_t *)(p + ORG - (o & 3)), o & 3};
    }
    // 8 bytes at p + ORG + off, off a multiple of 4 (the shift stays sh)
    __device__ __forceinline__ uint2 u64(int off) const {
        const uint32_t *q = qa + off / 4;
        const uint32_t d0 = q[0], d1 = q[1], d2 = q[2];
        return make_uint2(__builtin_amdgcn_alignbyte(d1, d0, sh), __builtin_amdgcn_alignbyte(d2, d1, sh));
    }
    // 4 bytes at p + ORG + off, off a multiple of 4
    __device__ __forceinline__ uint32_t u32(int off) const {
        const uint32_t *q = qa + off / 4;
        return __builtin_amdgcn_alignbyte(q[1], q[0], sh);
    }
    // 4 bytes at p + ORG + off, any off
    __device__ __forceinline__ uint32_t u32x(int off) const {
        const uint32_t t = sh + (uint32_t)off;
        const uint32_t *q = qa + (t >> 2);
        return __builtin_amdgcn_alignbyte(q[1], q[0], t & 3);
    }
    // 8 bytes at p + ORG + off, any off
    __device__ __forceinline__ uint2 u64x(int off) const {
        const uint32_t t = sh + (uint32_t)off, a = t & 3;
        const uint32_t *q = qa + (t >> 2);
        const uint32_t d0 = q[0], d1 = q[1], d2 = q[2];
        return make_uint2(__builtin_amdgcn_alignbyte(d1, d0, a), __builtin_amdgcn_alignbyte(d2, d1, a));
    }
};

// Lane-owned sub-blocks (SB): the K order of a super-block is permuted so that lane group grp owns
// sub-blocks grp and 4 + grp: K-step kk = 4 j + l takes octet l of sub-block 4 j + grp in K positions
// 8 grp .. 8 grp + 7 (the activations are packed in that order: k_order). A lane then reads its two
// sub-blocks' indices, signs and scales once per stage, and their scale's multiplier is worked out once
// for four fragments, instead of every lane group reading and unpacking every sub-block: about 18 VALU
// instructions per fragment instead of 28 (IQ2_XXS). Layers of 256 IQ2 experts, top-8, 2048 x 512: 64
// tokens 174 -> 159 us, 1,500 tokens 253 -> 238; 128 Q4_K experts, 768 x 2048, 256 tokens 181 -> 158; dense
// Q4_K 4096 x 4096 at 512 rows 54.8 -> 51.2.
//
// Traits common to the formats: KST K-steps per stage; SCALE 0 = one f16 scale per super-block
// (read by scale()), 1 = MXFP4's power-of-two block scales, 2 = one f16 scale per 32-weight block
// (read by step_scale()).
struct MIQ2_XXS {
    static constexpr int TS = 66, SBK = 256, LDS = 256 * 16;
    static constexpr int KST = 8, SCALE = 0, ORG = 2;
    static constexpr bool SB = true;
    static __device__ void fill(uint8_t *lds, int tid, int nt) { copy_tab(lds, c_iq2xxs_f16, tid, nt); }
    // A fragment is the grid entry (one lookup) with the signs applied arithmetically: the 7 sign
    // bits of the octet plus their even parity as the 8th (ksigns_iq2xs; apply_signs ignores the
    // popcount's higher bits), and the multiplier 8*(2s+1) as one packed multiply, exact in fp16 with
    // the grid values (at most 43*248 = 1333*8); d takes the 8 back out. A super-block scale of 0
    // gives the multiplier 0: its codes must not contribute.
    struct Stage {
        uint2 q[2];
        uint32_t mul[2];
        float d;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            d = h2f(lds_u16(w.p)) * (0.125f / 8);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                q[j] = w.u64(8 * grp + 32 * j);
                mul[j] = splat_mult(d == 0.f ? 0u : ((q[j].y >> 28) << 4) | 8);
            }
        }
    };
    struct Raw {};
    struct Look { uint4 g; };
    static __device__ __forceinline__ Raw raw(const WinRef &, const Stage &, int, int) { return Raw{}; }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &st, int kk, int, const uint8_t *lds, bool) {
        return Look{((const uint4 *)lds)[(st.q[kk >> 2].x >> (8 * (kk & 3))) & 0xFF]};
    }
    static __device__ __forceinline__ uint4 make(const Raw &, const Look &l, const Stage &st, int kk, int, bool) {
        const uint32_t s7 = (st.q[kk >> 2].y >> (7 * (kk & 3))) & 127;
        return scale4(apply_signs(l.g, s7 | ((uint32_t)__builtin_popcount(s7) << 7)), st.mul[kk >> 2]);
    }
};

struct MIQ2_S {
    static constexpr int TS = 82, SBK = 256, LDS = 1024 * 16;
    static constexpr int KST = 8, SCALE = 0, ORG = 2;
    static constexpr bool SB = true;
    static __device__ void fill(uint8_t *lds, int tid, int nt) { copy_tab(lds, c_iq2s_f16, tid, nt); }
    // index bytes, sign bytes, high index bits of the lane's sub-blocks; the multipliers 8*(2s+1) of their
    // halves, as (s << 4) | 8 (d takes the 8 back out)
    struct Stage {
        uint32_t qs[2], sg[2], qh[2], mul[2][2];
        float d;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            d = h2f(lds_u16(w.p)) * (0.125f / 8);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                qs[j] = w.u32(4 * grp + 16 * j);
                sg[j] = w.u32(32 + 4 * grp + 16 * j);
                qh[j] = lds_u8(w.p + 66 + grp + 4 * j);
                const uint32_t s = lds_u8(w.p + 74 + grp + 4 * j);
                mul[j][0] = splat_mult(d == 0.f ? 0u : ((s << 4) & 0xF0) | 8);
                mul[j][1] = splat_mult(d == 0.f ? 0u : (s & 0xF0) | 8);
            }
        }
    };
    struct Raw {};
    struct Look { uint4 g; };
    static __device__ __forceinline__ Raw raw(const WinRef &, const Stage &, int, int) { return Raw{}; }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &st, int kk, int, const uint8_t *lds, bool) {
        const int j = kk >> 2, l = kk & 3;
        return Look{((const uint4 *)lds)[((st.qs[j] >> (8 * l)) & 0xFF) | (((st.qh[j] >> (2 * l)) & 3) << 8)]};
    }
    static __device__ __forceinline__ uint4 make(const Raw &, const Look &l, const Stage &st, int kk, int, bool) {
        const int j = kk >> 2;
        return scale4(apply_signs(l.g, (st.sg[j] >> (8 * (kk & 3))) & 0xFF), st.mul[j][(kk >> 1) & 1]);
    }
};

struct MIQ3_S {
    static constexpr int TS = 110, SBK = 256, LDS = 512 * 8;
    static constexpr int KST = 8, SCALE = 0, ORG = 2;
    static constexpr bool SB = true;
    static __device__ void fill(uint8_t *lds, int tid, int nt) { copy_tab(lds, c_iq3s_f16, tid, nt); }  // entry i: 4 halves at byte 8*i
    // as MIQ2_S, two 4-value entries per octet and one multiplier 8*(2s+1) per sub-block
    struct Stage {
        uint2 qs[2];
        uint32_t sg[2], qh[2], mul[2];
        float d;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            d = h2f(lds_u16(w.p)) * 0.125f;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                qs[j] = w.u64(8 * grp + 32 * j);
                sg[j] = w.u32(72 + 4 * grp + 16 * j);
                qh[j] = lds_u8(w.p + 66 + grp + 4 * j);
                const uint32_t s = (uint32_t)lds_u8(w.p + 106 + (grp >> 1) + 2 * j) >> (4 * (grp & 1));
                mul[j] = splat_mult(d == 0.f ? 0u : ((s << 4) & 0xF0) | 8);
            }
        }
    };
    struct Raw {};
    struct Look { uint2 x, y; };
    static __device__ __forceinline__ Raw raw(const WinRef &, const Stage &, int, int) { return Raw{}; }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &st, int kk, int, const uint8_t *lds, bool) {
        const int j = kk >> 2, l = kk & 3;
        const uint32_t q = (l < 2 ? st.qs[j].x : st.qs[j].y) >> (16 * (l & 1)), h = st.qh[j] >> (2 * l);
        const uint2 *g = (const uint2 *)lds;
        return Look{g[(q & 0xFF) | ((h & 1) << 8)], g[((q >> 8) & 0xFF) | ((h & 2) << 7)]};
    }
    static __device__ __forceinline__ uint4 make(const Raw &, const Look &l, const Stage &st, int kk, int, bool) {
        const int j = kk >> 2;
        return scale4(apply_signs(make_uint4(l.x.x, l.x.y, l.y.x, l.y.y), (st.sg[j] >> (8 * (kk & 3))) & 0xFF), st.mul[j]);
    }
};

// MXFP4: one scale (e8m0) per 32 weights, so per K-step. The fragment carries the power of two
// 2^(e - base) relative to the largest exponent of the row's stage, and the accumulator is
// rescaled when that base changes; in fp16 the product code * 2^(e - base) is exact down to
// 2^-24 of the stage's largest block scale (smaller contributions round).

struct MMXFP4 {
    static constexpr int TS = 17, SBK = 32, LDS = 0;
    static constexpr int KST = 8, SCALE = 1, ORG = 1;
    static constexpr bool SB = false;
    static __device__ void fill(uint8_t *, int, int) {}
    struct Stage {
        __device__ __forceinline__ void load(const WinRef &, int) {}
    };
    static __device__ __forceinline__ uint32_t expo(const uint8_t *win, int kk) { return lds_u8(win + TS * kk); }
    // Lane group grp takes bytes 4grp..4grp+3 of the block, both nibbles of each: weights 4grp+i
    // and 4grp+i+16 (the low and high nibbles of byte 4grp+i) at fragment positions 2i, 2i+1.
    // The K order of a 32-weight step is thus permuted; the activations are packed in the same
    // order (K_PAIRS), so every product pairs the same weight
    // and activation as in natural order.
    struct Raw { uint32_t q; uint32_t e; };
    struct Look {};
    static __device__ __forceinline__ Raw raw(const WinRef &w, const Stage &, int kk, int grp) {
        return Raw{w.u32x(TS * kk + 4 * grp), expo(w.p, kk)};
    }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &, int, int, const uint8_t *, bool) { return Look{}; }
    // The fragment by gfx950's scaled FP4 conversion (v_cvt_scalef32_pk_f16_fp4: the two E2M1
    // values of one byte, low nibble first, times an f32 scale, to fp16), one conversion per byte
    // of the lane's dword: the scale 2^(de+1) gives the doubled E2M1 codes times 2^de, de = e - base
    // <= 0 the block's exponent against the stage's largest. Every product is exact in fp16 down
    // to 2^-24 of that largest block scale; below it, it rounds.
    static __device__ __forceinline__ uint32_t cvt2(uint32_t v, float sc, int sel) {
        f16x2 h;
        if (sel == 0)
            h = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 0);
        else if (sel == 1)
            h = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 1);
        else if (sel == 2)
            h = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 2);
        else
            h = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 3);
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ uint4 make_mx(const Raw &r, int, int de) {
        const float sc = de >= -127 ? __uint_as_float((uint32_t)(de + 128) << 23) : 0.f;
        return make_uint4(cvt2(r.q, sc, 0), cvt2(r.q, sc, 1), cvt2(r.q, sc, 2), cvt2(r.q, sc, 3));
    }
};

// 8 small unsigned byte values (v < 1024) of two dwords -> fp16 (1024 + v), by placing each byte
// under an 0x64 high byte
__device__ __forceinline__ uint4 bytes_plus_1024(uint32_t w0, uint32_t w1) {
    return make_uint4(__builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u),
                      __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u));
}
// x * mul + add on each fp16 pair (one rounding: exact when the result is a small integer)
__device__ __forceinline__ uint32_t pk_fma_u(uint32_t x, uint32_t mul, uint32_t add) {
    const f16x2 r = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, x), __builtin_bit_cast(f16x2, mul), __builtin_bit_cast(f16x2, add));
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint4 fma4(uint4 v, uint32_t mul, uint32_t add) {
    return make_uint4(pk_fma_u(v.x, mul, add), pk_fma_u(v.y, mul, add), pk_fma_u(v.z, mul, add), pk_fma_u(v.w, mul, add));
}
__device__ __forceinline__ uint32_t splat_f16f(float v) {
    const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)v);
    return h | (h << 16);
}

// Q8_0: codes are the int8 quants themselves (exact in fp16), one f16 scale per block (per K-step)
struct MQ8_0 {
    static constexpr int TS = 34, SBK = 32, LDS = 16;
    static constexpr int KST = 4, SCALE = 2, ORG = 2;
    static constexpr bool SB = false;
    static __device__ void fill(uint8_t *, int, int) {}
    struct Stage {
        __device__ __forceinline__ void load(const WinRef &, int) {}
    };
    // (q + 128) + 1024 from the byte pattern, then x - 1152 (or 0 when the block's scale is 0)
    struct Raw { uint2 q; float d; };
    struct Look {};
    static __device__ __forceinline__ Raw raw(const WinRef &w, const Stage &, int kk, int grp) {
        return Raw{w.u64x(TS * kk + 8 * grp), h2f(lds_u16(w.p + TS * kk))};
    }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &, int, int, const uint8_t *, bool) { return Look{}; }
    static __device__ __forceinline__ float step_scale(const Raw &r) { return r.d; }
    static __device__ __forceinline__ uint4 make(const Raw &r, const Look &, const Stage &, int, int, bool zero) {
        const uint4 x = bytes_plus_1024(r.q.x ^ 0x80808080u, r.q.y ^ 0x80808080u);
        const uint32_t one = zero ? 0u : 0x3C003C00u, off = zero ? 0u : 0xE480E480u;  // 1.0, -1152.0
        return fma4(x, one, off);
    }
};

// Q4_K: y = d*sc*q - dmin*m per sub-block of 32 (k_quants.rs:1821-1849, get_scale_min_k4 in
// quantized/utils.rs:50-60).
struct MQ4_K {
    static constexpr int TS = 144, SBK = 256, LDS = 16;
    static constexpr int KST = 8, SCALE = 0, ORG = 16;
    static constexpr bool SB = true;
    static __device__ void fill(uint8_t *, int, int) {}
    // The minimum term is folded into the codes: y = s (a q - b) per weight, with the running
    // scale s = max(|d|, |dmin|) of the super-block, a = (d / s) sc and b = (dmin / s) m of the
    // sub-block (both within 63 in magnitude, so fp16 keeps them to 2^-11 of themselves, and the
    // code a q - b takes one rounding). One accumulator and one MFMA per weight fragment.
    static __device__ __forceinline__ float s_of(float d, float dm) { return fmaxf(fabsf(d), fabsf(dm)); }
    // s, and the fp16 pairs a and -b of the lane's sub-blocks (0 where s is 0)
    struct Stage {
        uint32_t a[2], b[2];
        float d;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            const uint2 lo = w.u64(-12);  // scale bytes 0..7, then 8..11
            const int sh = 8 * grp;
            const uint32_t b0 = (lo.x >> sh) & 0xFF, b1 = (lo.y >> sh) & 0xFF, b2 = (w.u32(-4) >> sh) & 0xFF;
            const uint32_t dd = w.u32(-16);  // d, then dmin
            const float d0 = h2f(dd & 0xFFFFu), dm = h2f(dd >> 16);
            d = s_of(d0, dm);
            const float r = d > 0.f ? __builtin_amdgcn_rcpf(d) : 0.f, fd = d0 * r, fm = dm * r;
            // sub-block grp: the low 6 bits; 4 + grp: a nibble, and the top 2 bits of byte grp (get_scale_min_k4)
            a[0] = splat_f16f(fd * (float)(b0 & 63));
            b[0] = splat_f16f(-fm * (float)(b1 & 63));
            a[1] = splat_f16f(fd * (float)((b2 & 0xF) | ((b0 >> 6) << 4)));
            b[1] = splat_f16f(-fm * (float)((b2 >> 4) | ((b1 >> 6) << 4)));
        }
    };
    // codes a q - b of octet kk & 3 (sub-blocks 2c, 2c+1 are the low and high nibbles of qs[32c..32c+32))
    struct Raw { uint2 q; };
    struct Look {};
    static __device__ __forceinline__ Raw raw(const WinRef &w, const Stage &, int kk, int grp) {
        return Raw{w.u64(64 * (kk >> 2) + 32 * (grp >> 1) + 8 * (kk & 3))};
    }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &, int, int, const uint8_t *, bool) { return Look{}; }
    static __device__ __forceinline__ uint4 make(const Raw &r, const Look &, const Stage &st, int kk, int grp, bool) {
        const int sh = 4 * (grp & 1);
        // q as fp16 (1024 + q less 1024: exact), then a q - b
        const uint4 x = fma4(bytes_plus_1024((r.q.x >> sh) & 0x0F0F0F0Fu, (r.q.y >> sh) & 0x0F0F0F0Fu), splat_f16f(1.0f),
                             splat_f16f(-1024.0f));
        return fma4(x, st.a[kk >> 2], st.b[kk >> 2]);
    }
};

// Q2_K (what the shrink writes): y = d*(sc&15)*q - dmin*(sc>>4) per 16 weights (k_quants.rs:1152-1190).
// Sub-block 4j + grp is bits 2 grp of qs[32j ..), its halves scaled by bytes 8j + 2 grp and the next.
// The minimum term folded into the codes as for Q4_K: y = s (a q - b), s = max(|d|, |dmin|),
// a = (d / s) (sc & 15), b = (dmin / s) (sc >> 4), both within 15 in magnitude.
struct MQ2_K {
    static constexpr int TS = 84, SBK = 256, LDS = 16;
    static constexpr int KST = 8, SCALE = 0, ORG = 16;
    static constexpr bool SB = true;
    static __device__ void fill(uint8_t *, int, int) {}
    struct Stage {
        uint32_t a[2][2], b[2][2];  // per sub-block of the lane and half
        float d;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            const uint32_t dd = w.u32(64);  // d, then dmin
            const float d0 = h2f(dd & 0xFFFFu), dm = h2f(dd >> 16);
            d = MQ4_K::s_of(d0, dm);
            const float r = d > 0.f ? __builtin_amdgcn_rcpf(d) : 0.f, fd = d0 * r, fm = dm * r;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t sb = w.u32(-16 + 8 * j + 4 * (grp >> 1)) >> (16 * (grp & 1));
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    a[j][h] = splat_f16f(fd * (float)((sb >> (8 * h)) & 0xF));
                    b[j][h] = splat_f16f(-fm * (float)((sb >> (8 * h + 4)) & 0xF));
                }
            }
        }
    };
    struct Raw { uint2 q; };
    struct Look {};
    static __device__ __forceinline__ Raw raw(const WinRef &w, const Stage &, int kk, int) { return Raw{w.u64(32 * (kk >> 2) + 8 * (kk & 3))}; }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &, int, int, const uint8_t *, bool) { return Look{}; }
    static __device__ __forceinline__ uint4 make(const Raw &r, const Look &, const Stage &st, int kk, int grp, bool) {
        const int sh = 2 * grp, j = kk >> 2, h = (kk >> 1) & 1;
        const uint4 x = fma4(bytes_plus_1024((r.q.x >> sh) & 0x03030303u, (r.q.y >> sh) & 0x03030303u), splat_f16f(1.0f),
                             splat_f16f(-1024.0f));
        return fma4(x, st.a[j][h], st.b[j][h]);
    }
};

// IQ3_XXS: octet l of sub-block ib is the grid entries qs[8ib + 2l], qs[8ib + 2l + 1] (4 values each) with
// the signs of index (w >> 7l) & 127, w the sub-block's word at byte 66 + 4ib (scale nibble s on top). The
// multiplier 8*(2s+1), as (s << 4) | 8, keeps the codes (at most 8*31*62) exact in fp16; d takes the 8 and
// the 1/4 of dl = d*(2s+1)/4 back out.
struct MIQ3_XXS {
    static constexpr int TS = 98, SBK = 256, LDS = 256 * 8;
    static constexpr int KST = 8, SCALE = 0, ORG = 2;
    static constexpr bool SB = true;
    static __device__ void fill(uint8_t *lds, int tid, int nt) { copy_tab(lds, c_iq3xxs_f16, tid, nt); }  // entry i: 4 halves at byte 8*i
    struct Stage {
        uint2 qs[2];
        uint32_t w[2], mul[2];
        float d;
        __device__ __forceinline__ void load(const WinRef &win, int grp) {
            d = h2f(lds_u16(win.p)) * (0.25f / 8);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                qs[j] = win.u64(8 * grp + 32 * j);
                w[j] = win.u32(64 + 4 * grp + 16 * j);
                mul[j] = splat_mult(d == 0.f ? 0u : ((w[j] >> 28) << 4) | 8);
            }
        }
    };
    struct Raw {};
    struct Look { uint2 x, y; };
    static __device__ __forceinline__ Raw raw(const WinRef &, const Stage &, int, int) { return Raw{}; }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &st, int kk, int, const uint8_t *lds, bool) {
        const int j = kk >> 2, l = kk & 3;
        const uint32_t q = (l < 2 ? st.qs[j].x : st.qs[j].y) >> (16 * (l & 1));
        const uint2 *g = (const uint2 *)lds;
        return Look{g[q & 0xFF], g[(q >> 8) & 0xFF]};
    }
    static __device__ __forceinline__ uint4 make(const Raw &, const Look &l, const Stage &st, int kk, int, bool) {
        const uint32_t s7 = (st.w[kk >> 2] >> (7 * (kk & 3))) & 127;
        return scale4(apply_signs(make_uint4(l.x.x, l.x.y, l.y.x, l.y.y), s7 | ((uint32_t)__builtin_popcount(s7) << 7)), st.mul[kk >> 2]);
    }
};

// IQ4_XS: K-step kk is sub-block kk, with its own scale d*(ls - 32) (per K-step, as Q8_0). Lane
// group grp takes the low (grp < 2) or high nibbles of qs[16kk + 8(grp&1) ..); a nibble's level
// kvalues[n] (exact in fp16) comes from a byte table of kvalues + 128 by two byte permutes and a
// select on the nibble's top bit, then through the fp16 1024 + byte pattern less 1152.
struct MIQ4_XS {
    static constexpr int TS = 136, SBK = 256, LDS = 16;
    static constexpr int KST = 8, SCALE = 2, ORG = 0;
    static constexpr bool SB = false;
    static __device__ void fill(uint8_t *, int, int) {}
    // d | scales_h << 16 and scales_l[4]: the super-block's first 8 bytes, read once per stage
    struct Stage {
        uint32_t h0, h1;
        __device__ __forceinline__ void load(const WinRef &w, int) {
            const uint2 h = w.u64(0);
            h0 = h.x;
            h1 = h.y;
        }
    };
    struct Raw { uint2 q; float d; };
    struct Look {};
    static __device__ __forceinline__ Raw raw(const WinRef &w, const Stage &st, int kk, int grp) {
        const uint32_t ls = ((st.h1 >> (4 * kk)) & 0xF) | (((st.h0 >> (16 + 2 * kk)) & 3) << 4);
        return Raw{w.u64(8 + 16 * kk + 8 * (grp & 1)), h2f(st.h0 & 0xFFFF) * (float)((int)ls - 32)};
    }
    static __device__ __forceinline__ Look look(const Raw &, const Stage &, int, int, const uint8_t *, bool) { return Look{}; }
    static __device__ __forceinline__ float step_scale(const Raw &r) { return r.d; }
    // kvalues_iq4nl + 128 as bytes, entries 0..15 over four dwords
    static constexpr uint32_t T0 = 0x3F2D1801u, T1 = 0x766A5D4Fu, T2 = 0xA6998D81u, T3 = 0xF1D9C5B5u;
    static __device__ __forceinline__ uint32_t levels4(uint32_t n) {  // 4 nibbles (one per byte) -> 4 table bytes
        const uint32_t lo = __builtin_amdgcn_perm(T1, T0, n & 0x07070707u);
        const uint32_t hi = __builtin_amdgcn_perm(T3, T2, n & 0x07070707u);
        const uint32_t top = ((n >> 3) & 0x01010101u) * 0xFFu;
        return (hi & top) | (lo & ~top);
    }
    static __device__ __forceinline__ uint4 make(const Raw &r, const Look &, const Stage &, int, int grp, bool zero) {
        const int sh = 4 * (grp >> 1);
        const uint4 x = bytes_plus_1024(levels4((r.q.x >> sh) & 0x0F0F0F0Fu), levels4((r.q.y >> sh) & 0x0F0F0F0Fu));
        const uint32_t one = zero ? 0u : 0x3C003C00u, off = zero ? 0u : 0xE480E480u;  // 1.0, -1152.0
        return fma4(x, one, off);
    }
};

// A stage is KST K-steps (8: 256 weights of k; 4 for Q8_0). The window of a row for a stage
// holds the stage's bytes (an IQ, Q2_K or Q4_K super-block, or KST MXFP4 / Q8_0 blocks) from the
// 16-byte boundary at or below their start, in PCS pieces of 16 bytes. PCS is odd: the 16 rows of
// a fragment read their windows at a stride of 4*PCS dwords, and an even PCS put rows 8 (or 4)
// apart on the same LDS banks (config 4 prefill 1,302-1,310 -> 1,253-1,261 us, config 3 271-275 ->
// 267-268, the last piece a re-load nothing reads).
template <class MF>
struct Win {
    static constexpr int SEG = MF::SBK == 32 ? MF::KST * MF::TS : MF::TS;
    static constexpr int PCS = ((SEG + (MF::TS % 2 ? 15 : 14) + 15) / 16) | 1;
    static constexpr int BYTES = 16 * PCS;
};

// ------------------------------------------------------------------------------ kernels

template <int V> struct Ic { static constexpr int value = V; };

__device__ __forceinline__ f16x8 as_f16x8(uint4 v) { return __builtin_bit_cast(f16x8, v); }

// Direct global-to-LDS loads, without passing through registers: lane l of the wave writes 16 (or 4)
// bytes at an LDS address, the same for the whole wave, + 16 l (4 l). Issued as inline asm instead of
// through __builtin_amdgcn_global_load_lds: the compiler counts the builtin as an LDS store that any later
// LDS read at a dynamic address (a table lookup) may alias, and puts an s_waitcnt vmcnt(0) before that
// read, so every prefetch is waited for right after it is issued. A kernel orders these loads itself: an
// explicit s_waitcnt on the issuing wave, then a barrier, before any wave reads the bytes, and a barrier
// between the last read of a buffer and the loads that overwrite it. Loads return in order, so the
// compiler's own vmcnt waits stay correct with these in flight (they only wait longer: a register spill's
// reload then waits for the prefetches before it).
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)p);
}
// base: wave-uniform; off: the lane's 32-bit offset
__device__ __forceinline__ void dma16_s(const uint8_t *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
// g: the lane's address
__device__ __forceinline__ void dma16(const void *g, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void *g, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(lds) : "memory", "m0");
}

// The end of a split-K work item (MODE 2), its partial rows stored: the last block to get here sums them.
template <int RPB, int NT>
__device__ __forceinline__ void split_sum(const MfArgs &a, int item, int nblk, int tile_m, const int *meta_pick, int tid, int *split_last) {
    // The last of the item's splits to get here adds the partial rows in split order (as a
    // separate pass over all of them would): the partial stores are at the coherence
    // point once this thread's stores have completed, before the block's arrival.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0)
        *split_last = __hip_atomic_fetch_add(a.split_cnt + item, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                     (int)gridDim.y - 1;
    __syncthreads();
    if (*split_last) {
        // partial values read at the coherence point (buffer loads with the sc1 policy,
        // the form of an agent-scope load), 8 splits in flight at a time
        const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)a.dn, (short)0, (int)(gridDim.y * a.split_stride * 4), 0x00020000);
        const int cols = min(RPB, a.n - nblk * RPB), nsp = (int)gridDim.y;
        for (int e = tid; e < tile_m * cols; e += NT) {
            const int r = e / cols, n = nblk * RPB + (e - r * cols);
            const int o = (int)((int64_t)meta_pick[r] * a.n + n);
            float acc = 0.f;
            for (int s0 = 0; s0 < nsp; s0 += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++)  // past the last split: 0 from the buffer's range, unused
                    v[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(pr, 4 * (o + (s0 + u) * (int)a.split_stride), 0, 16));
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (s0 + u < nsp) acc = (s0 + u == 0) ? v[u] : acc + v[u];
            }
            a.y[o] = acc;
        }
    }
}

// What a pack launch does besides (PackExtra): tile i of a dense matmul (rows MF_MT i .., "slot" 0) and
// the zeroed split counters.
__device__ __forceinline__ void pack_extra(const PackExtra &e) {
    if (e.tiles && blockIdx.x == 0) {
        const int nt = (e.m + MF_MT - 1) / MF_MT;
        for (int i = threadIdx.x; i < nt; i += blockDim.x) e.tiles[i] = MfTile{0, i * MF_MT, min(MF_MT, e.m - i * MF_MT), 0};
        if (threadIdx.x == 0) *e.n_tiles = nt;
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < e.n_zero; i += gridDim.x * blockDim.x) e.zero[i] = 0;
}

}  // namespace cw
