// Grouped and dense GEMMs at f32 accuracy on the fp16 matrix instruction (gfx950), for the formats whose
// other path is one f32 matvec per row of x: Q5_K and Q6_K, and the formats they share a layer with.
//
// Every activation goes in as two fp16 terms under a power of two per super-block of its row, hi = fp16(x)
// and lo = fp16((x - hi) 2^12), which together hold x to 2^-23 of itself, and values below 2^-29 of the
// super-block's largest to 2^-52 of that. The weight codes are numbers that fp16 holds exactly: sc (q - C) / 2
// of Q4_K and Q5_K (C the middle of q's range), Q8_0's quants; Q6_K's sc (q - 32) reaches 4,096 and goes
// in as its fp16 rounding and the exact rest (0 or +-1). A product then is two matrix instructions per
// fragment (three for Q6_K, whose rest times lo is below 2^-23 of the product), hi and what is below it in
// accumulators of their own: an instruction rounds its accumulator every 8 products, at the size of its sums,
// so the small terms cost the large ones nothing. The minimum term of Q4_K and Q5_K and what C took off are a
// ninth K-step per super-block: codes m and C sc against the sub-blocks' sums of x, which the pack takes in
// f64 and holds in three terms, so that what all weights of a sub-block have in common meets x exactly.
// A super-block's sum is scaled into a further accumulator set in f32, so no running scale's rounding is
// carried through a row. Error against f64 (rel-L2; the matvec's, then with one scale and one accumulator per
// row and uncentred codes): Q5_K 513 x 4096 at 77 rows 1.08e-7 (1.35, 1.75), Q6_K 1.35e-7 (2.15, 1.69); layers
// of 4 experts, 15 tokens, 4096 x 512: Q8_0 / Q4_K 2.1e-7 (2.4, 8.0), Q4_K / Q8_0 2.1e-7 (2.3, 3.0), Q5_K /
// Q6_K 2.1e-7 (3.9, 3.1), Q4_K alone 0.9e-7 (0.8, 1.2).
#include <math.h>

#include <atomic>

#include "cw_common.h"
#include "cw_gmm_dev.h"
#include "cw_mfma.h"
#include "cw_wave.h"

namespace cw {

// ------------------------------------------------------------------------------ formats
// Per format: NF code fragments per K-step of 32 weights (lane group grp: weights 8 grp .. 8 grp + 7),
// MIN the step of the sums, STEP a scale per K-step instead of one per super-block (stage). Stage holds
// what a lane needs of its row for the whole stage; w is the row's window from the stage's first byte.

// the terms' second halves are held times LO (k_pack_split)
constexpr float LO = 4096.0f;
constexpr uint32_t LO_F16X2 = 0x6C006C00u, LO_INV_F16X2 = 0x0C000C00u;  // LO and 1 / LO, twice each

// half i of an fp16 pair, twice (an operand select of the packed instruction that takes it)
__device__ __forceinline__ uint32_t splat_half(uint32_t v, int i) {
    const f16x2 h = __builtin_bit_cast(f16x2, v);
    return __builtin_bit_cast(uint32_t, f16x2{h[i], h[i]});
}
// sc (q - C) / 2 for q < 64, from s2 = sc / 2 twice: the bytes q + 64 - C under 0x64 are 1088 + q - C, and
// 544 sc is exact in fp16 (17 times a 6-bit number), as is every code (at most 10 bits and a half)
template <int C>
__device__ __forceinline__ uint4 codes_centred(uint32_t q0, uint32_t q1, uint32_t s2) {
    constexpr uint32_t off = 0x01010101u * (64 - C);
    return fma4(bytes_plus_1024(q0 + off, q1 + off), s2, pk_mul_u(s2, 0xE440E440u));  // -1088
}
// What Q4_K and Q5_K share: d, dmin and the 12 bytes of eight 6-bit scales and minima (get_scale_min_k4)
struct K4Stage {
    uint32_t s2[4];  // half of the scales of sub-blocks 2i and 2i + 1, fp16
    __device__ __forceinline__ void load_scales(const WinRef &w) {
        const uint32_t b0 = w.u32(4), b2 = w.u32(12);
        const uint4 x = fma4(bytes_plus_1024(b0 & 0x3F3F3F3Fu, (b2 & 0x0F0F0F0Fu) | ((b0 >> 2) & 0x30303030u)), 0x38003800u, 0xE000E000u);  // (x - 1024) / 2
        s2[0] = x.x;
        s2[1] = x.y;
        s2[2] = x.z;
        s2[3] = x.w;
    }
    // the codes that meet the sub-blocks' sums of x over 32, times one: the minima, and the scales' halves
    // times 32 C for what the centre took off the codes
    template <int C>
    __device__ __forceinline__ void sums_codes(const WinRef &w, float one, f16x8 &mins, f16x8 &scs) const {
        const uint32_t b1 = w.u32(8), b2 = w.u32(12), f = splat_f16f(32.f * C * one);
        mins = as_f16x8(fma4(bytes_plus_1024(b1 & 0x3F3F3F3Fu, ((b2 >> 4) & 0x0F0F0F0Fu) | ((b1 >> 2) & 0x30303030u)), splat_f16f(one),
                             splat_f16f(-1024.f * one)));
        scs = as_f16x8(scale4(make_uint4(s2[0], s2[1], s2[2], s2[3]), f));
    }
    // d for codes that are halves, dmin for sums over 32
    static __device__ __forceinline__ void scales(const WinRef &w, float &d, float &dm) {
        const uint32_t dd = w.u32(0);
        d = 2.f * h2f(dd & 0xFFFFu);
        dm = -32.f * h2f(dd >> 16);
    }
};

struct SQ4_K {
    static constexpr int TS = 144, SBK = 256, NF = 1, C = 8;
    static constexpr bool MIN = true, STEP = false;
    struct Stage : K4Stage {
        __device__ __forceinline__ void load(const WinRef &w, int) { load_scales(w); }
    };
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &st, int kk, int grp, uint4 (&f)[1]) {
        const uint2 q = w.u64(16 + 32 * (kk >> 1) + 8 * grp);
        const int sh = 4 * (kk & 1);
        f[0] = codes_centred<C>((q.x >> sh) & 0x0F0F0F0Fu, (q.y >> sh) & 0x0F0F0F0Fu, splat_half(st.s2[kk >> 1], kk & 1));
        return 0.f;
    }
};

struct SQ5_K {
    static constexpr int TS = 176, SBK = 256, NF = 1, C = 16;
    static constexpr bool MIN = true, STEP = false;
    struct Stage : K4Stage {
        uint2 h;  // the lane's bytes of qh: bit kk is weight kk's fifth
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            load_scales(w);
            h = w.u64(16 + 8 * grp);
        }
    };
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &st, int kk, int grp, uint4 (&f)[1]) {
        const uint2 q = w.u64(48 + 32 * (kk >> 1) + 8 * grp);
        const int sh = 4 * (kk & 1);
        f[0] = codes_centred<C>(((q.x >> sh) & 0x0F0F0F0Fu) | (((st.h.x >> kk) & 0x01010101u) << 4),
                                ((q.y >> sh) & 0x0F0F0F0Fu) | (((st.h.y >> kk) & 0x01010101u) << 4), splat_half(st.s2[kk >> 1], kk & 1));
        return 0.f;
    }
};

struct SQ6_K {
    static constexpr int TS = 210, SBK = 256, NF = 2;
    static constexpr bool MIN = false, STEP = false;
    struct Stage {
        uint32_t sc[4];  // the scales of the lane's half of K-steps 2i and 2i + 1, fp16
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            const uint2 a = w.u64(192), b = w.u64(200);
            const int sh = 8 * (grp >> 1);
            const uint32_t v[4] = {a.x, a.y, b.x, b.y};
#pragma unroll
            for (int i = 0; i < 4; i++)  // (s + 128) + 1024, less 1152
                sc[i] = pk_fma_u((((v[i] >> sh) & 0x00FF00FFu) ^ 0x00800080u) | 0x64006400u, 0x3C003C00u, 0xE480E480u);
        }
    };
    static __device__ __forceinline__ float scale(const WinRef &w) { return h2f(w.u32(208) & 0xFFFFu); }
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &st, int kk, int grp, uint4 (&f)[2]) {
        const int h = kk >> 2, r = kk & 3;
        const uint2 l = w.u64(64 * h + 32 * (r & 1) + 8 * grp), g = w.u64(128 + 32 * h + 8 * grp);
        const int sh = 4 * (r >> 1);
        const uint32_t q0 = ((l.x >> sh) & 0x0F0F0F0Fu) | (((g.x >> (2 * r)) & 0x03030303u) << 4);
        const uint32_t q1 = ((l.y >> sh) & 0x0F0F0F0Fu) | (((g.y >> (2 * r)) & 0x03030303u) << 4);
        const uint32_t sc = splat_half(st.sc[kk >> 1], kk & 1);
        const uint4 c = fma4(bytes_plus_1024(q0, q1), 0x3C003C00u, 0xE420E420u);  // 1.0, -1056.0: q - 32
        f[0] = scale4(c, sc);
        // the rest of the product, c sc - fp16(c sc), exact, 0 or +-1; times LO, beside the lo terms
        auto rest = [&](uint32_t x, uint32_t p) __attribute__((always_inline)) {
            const f16x2 n = -__builtin_bit_cast(f16x2, p);
            return pk_mul_u(pk_fma_u(x, sc, __builtin_bit_cast(uint32_t, n)), LO_F16X2);
        };
        f[1] = make_uint4(rest(c.x, f[0].x), rest(c.y, f[0].y), rest(c.z, f[0].z), rest(c.w, f[0].w));
        return 0.f;
    }
};

struct SQ8_0 {
    static constexpr int TS = 34, SBK = 32, NF = 1;
    static constexpr bool MIN = false, STEP = true;
    struct Stage {
        __device__ __forceinline__ void load(const WinRef &, int) {}
    };
    static __device__ __forceinline__ float scale(const WinRef &) { return 1.f; }
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &, int kk, int grp, uint4 (&f)[1]) {
        const uint2 q = w.u64x(TS * kk + 2 + 8 * grp);
        f[0] = fma4(bytes_plus_1024(q.x ^ 0x80808080u, q.y ^ 0x80808080u), 0x3C003C00u, 0xE480E480u);  // 1.0, -1152.0
        return h2f(w.u32x(TS * kk) & 0xFFFFu);
    }
};

// ------------------------------------------------------------------------------ kernel

// A block: 8 waves of 16 weight rows each (MODE 0: four on gate, four on up), one M-tile of up to MF_MT
// picks. A stage is 256 of k: the rows' windows (whole 16-byte pieces, as in cw_gmm_dev.h), then the
// activations in parts of KA K-steps, both terms, through two buffers: a part loads while the one before
// it is computed. Two blocks share a CU, so one's waits fall into the other's K-steps: with one window
// buffer a stage starts with a round trip to memory, and that is what bounds it (the waves wait 61 to 64 % of
// their time for loads and barriers, the matrix pipe is 9 to 17 % busy). Against a matvec per row
// or pick: Q6_K 4001 x 4096 at 77 rows 215 -> 34 us (pack included); a layer of 128 experts, top-8, Q4_K 768 x
// 2048 and Q6_K 2048 x 768 at 301 tokens 2.3 ms -> 0.22. What the small terms' own accumulators, the centred
// codes and the scales per super-block cost: nothing at few rows (Q5_K 4096 x 4096 at 77 rows 35 -> 34 us, the
// pack no longer one wave per row, and the 6-bit scales unpacked once per stage), 2 to 5 % at full tiles (Q6_K
// 4096 x 4096 at 512 rows 81 -> 84, a layer of 64 experts, Q5_K and Q6_K, 700 tokens 274 -> 288).
template <class SF, int MODE>
struct SpShape {
    static constexpr int KST = 8, NW = 8, NT = 64 * NW, NM = MODE == 0 ? 2 : 1, WPM = NW / NM, RPB = 16 * WPM;
    static constexpr int SEG = SF::SBK == 32 ? KST * SF::TS : SF::TS;
    static constexpr int PCS = ((SEG + 30) / 16) | 1, WB = 16 * PCS;  // pieces of a window (odd: LDS banks) and its bytes
    static constexpr int W_BYTES = NM * RPB * WB;
    static constexpr int KA = 2, PARTS = KST / KA + (SF::MIN ? 1 : 0);
    static constexpr int PART = KA * 2 * MF_MB * 1024, A_BYTES = 2 * PART;
    static constexpr int META = 2 * 128 * 4 + MF_MT * 4, PER_CU = 2;  // a stage's scales and the activation rows (by whole waves), picks
    static constexpr size_t lds_bytes() { return W_BYTES + A_BYTES + META; }
    static_assert(PER_CU * (W_BYTES + A_BYTES + META) <= 160 * 1024, "two blocks per CU");
    static_assert(MF_MT * RPB * 4 <= A_BYTES, "the gate/up exchange fits the activation buffers");
};

// MODE 0: gate and up with the activation, hidden rows in pile order; 1: down, a row per pick; 2: dense,
// split over K (see k_gmm, whose work items, tiles and epilogues these are).
template <class SF, int MODE>
__global__ __launch_bounds__(512, 4) void k_gms(const MfArgs a) {
    using S = SpShape<SF, MODE>;
    constexpr int KST = S::KST, KA = S::KA;
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int split_last;
    uint8_t *As = smem, *Ws = smem + S::A_BYTES;
    float *meta_sa = (float *)(Ws + S::W_BYTES);
    int *meta_row = (int *)(meta_sa + 128), *meta_pick = meta_row + 128;
    const int n_nb = (a.n + S::RPB - 1) / S::RPB, R = a.run_tiles, n_tiles = *a.n_tiles;
    const int n_ks = a.k / 32, n_st = (n_ks + KST - 1) / KST;
    const int st_lo = a.split_st ? blockIdx.y * a.split_st : 0, st_hi = a.split_st ? min(n_st, st_lo + a.split_st) : n_st;
    for (int item = blockIdx.x; item < a.n_items; item += gridDim.x) {
        const int run = item / (R * n_nb), b = item - run * R * n_nb;
        const int mt = run * R + (b & (R - 1)), nblk = b / R;
        if (mt >= n_tiles) continue;  // uniform across the block
        __syncthreads();              // every wave is done with the previous item's LDS
        // lane values from an opaque copy of the thread index: nothing derived from them is kept across items
        int tid = threadIdx.x;
        asm("" : "+v"(tid));
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = lane >> 4, l16 = lane & 15;
        const int mw = S::NM > 1 ? wave / S::WPM : 0, wrow = (wave - mw * S::WPM) * 16;  // this wave's matrix and its first row there
        const MfTile tile = a.tiles[mt];
        const int mbs = (tile.m + 15) >> 4;
        if (tid < tile.m) meta_pick[tid] = a.pile_pick ? a.pile_pick[tile.pos0 + tid] : tile.pos0 + tid;  // (the first stage's barriers publish it)
        // the first two waves bring a stage's scales, one per row of the tile (rows past the last: that one's; a
        // lane reads back its own)
        if (wave < 2) {
            const int pos = tile.pos0 + min(tid, tile.m - 1);
            meta_row[tid] = a.rows ? a.rows[pos] : pos;
        }
        // the activation row that this lane copies (pick block `wave`): hi at 0, lo at k, the sums at 2 k
        const bool stager = wave < mbs;
        const int apos = tile.pos0 + min(16 * wave + l16, tile.m - 1);
        const uint16_t *asrc = a.a16 + (int64_t)(a.rows ? a.rows[apos] : apos) * a.lda + 8 * grp;
        const uint8_t *wb0 = a.w0 + (int64_t)tile.slot * a.s0;
        const uint8_t *wb1 = S::NM > 1 ? a.w1 + (int64_t)tile.slot * a.s1 : wb0;
        auto row_off = [&](int r, int m) -> uint32_t {  // byte offset of block row r (of matrix m) within its matrix
            const int n = nblk * S::RPB + (r - m * S::RPB);
            return (uint32_t)(n < a.n ? n : 0) * (uint32_t)a.row_bytes;
        };
        const uint32_t as_lds = lds_addr(As), ws_lds = lds_addr(Ws), sa_lds = lds_addr(meta_sa);
        // windows as in k_gmm: each piece's row and place once per tile, 32-bit offsets from the 16-byte
        // boundary below the matrix
        constexpr int NP = S::NM * S::RPB * S::PCS, NTW = (NP + S::NT - 1) / S::NT;
        static_assert(S::RPB * S::PCS % 64 == 0, "a wave's pieces lie in one matrix");
        const uint32_t b0 = (uint32_t)(uintptr_t)wb0 & 15, b1 = (uint32_t)(uintptr_t)wb1 & 15;
        const uint8_t *wa0 = wb0 - b0, *wa1 = wb1 - b1;
        constexpr bool ALIGNED = SF::TS % 16 == 0;
        uint32_t wp_off[NTW], wp_p[NTW];
#pragma unroll
        for (int t = 0; t < NTW; t++) {
            const int w0 = S::NT * t + 64 * wave, i = (w0 < NP ? w0 : w0 - NP) + lane;
            const int r = i / S::PCS, m = S::NM > 1 ? __builtin_amdgcn_readfirstlane(r / S::RPB) : 0;
            wp_p[t] = (uint32_t)(i - r * S::PCS);
            wp_off[t] = row_off(r, m) + (m == 0 ? b0 : b1);
            if constexpr (ALIGNED) wp_off[t] = (wp_off[t] & ~15u) + 16 * min(wp_p[t], ((m == 0 ? b0 : b1) + S::SEG - 1) >> 4);
        }
        auto issue_w = [&](int st) __attribute__((always_inline)) {
            if (wave < 2) dma4(a.ascale + (int64_t)meta_row[tid] * n_st + st, sa_lds + 256 * wave);
            const uint32_t seg = SF::SBK == 32 ? SF::TS * min(KST, n_ks - st * KST) : SF::TS, at = (uint32_t)(S::SEG * st);
#pragma unroll
            for (int t = 0; t < NTW; t++) {
                const int w0 = S::NT * t + 64 * wave;
                if (w0 >= NP) break;  // uniform per wave: the last round's waves past the pieces
                uint32_t o = wp_off[t] + at;
                if constexpr (!ALIGNED) o = (o & ~15u) + 16 * min(wp_p[t], ((o & 15) + seg - 1) >> 4);
                dma16_s(S::NM > 1 && w0 >= S::RPB * S::PCS ? wa1 : wa0, o, ws_lds + 16 * w0);
            }
        };
        // this lane's row: its start in global memory mod 16
        const uint32_t lmis = (mw == 0 ? b0 : b1) + (ALIGNED ? 0 : row_off(mw * S::RPB + wrow + l16, mw));
        // part p of stage st: K-steps KA p .. (clamped to the row: unused), hi and lo; or the sums
        auto issue_a = [&](int st, int p, int buf) __attribute__((always_inline)) {
            if (!stager) return;
            const uint32_t dst = as_lds + buf * S::PART + wave * 1024;
            if (SF::MIN && p == KST / KA) {
                dma16(asrc + 2 * a.k + 32 * st, dst);
                return;
            }
#pragma unroll
            for (int kk = 0; kk < KA; kk++) {
                const int ks = SF::SBK == 32 ? min(st * KST + p * KA + kk, n_ks - 1) : st * KST + p * KA + kk;
                dma16(asrc + 32 * ks, dst + (2 * kk) * MF_MB * 1024);
                dma16(asrc + a.k + 32 * ks, dst + (2 * kk + 1) * MF_MB * 1024);
            }
        };

        f32x4 tot[MF_MB];
#pragma unroll
        for (int mb = 0; mb < MF_MB; mb++) tot[mb] = f32x4{0, 0, 0, 0};
        auto run_stages = [&](auto mbs_c) __attribute__((always_inline)) {
            constexpr int MBS = decltype(mbs_c)::value;
            int buf = 0;
            issue_a(st_lo, 0, 0);
            for (int st = st_lo; st < st_hi; st++) {
                if (st != st_lo) __syncthreads();  // every wave is done with the previous stage's windows
                issue_w(st);
                const int nk = min(KST, n_ks - st * KST);
                const WinRef w = WinRef::at<0>(Ws + (mw * S::RPB + wrow + l16) * S::WB + ((lmis + (uint32_t)(S::SEG * st)) & 15));
                typename SF::Stage stg;
                // hi times the codes, and (over LO) what is below it: lo times the codes and hi times Q6_K's rest.
                // With a scale per K-step: the stage's sum of both, scaled
                f32x4 acc[MBS], low[MBS];
#pragma unroll
                for (int p = 0; p < S::PARTS; p++) {
                    __builtin_amdgcn_s_waitcnt(0);  // this part's activations (and the windows and scales)
                    __syncthreads();
                    if (p + 1 < S::PARTS) issue_a(st, p + 1, buf ^ 1);
                    else if (st + 1 < st_hi) issue_a(st + 1, 0, buf ^ 1);
                    const uint8_t *A = As + buf * S::PART + lane * 16;
                    auto av = [&](int step, int term, int mb) __attribute__((always_inline)) {
                        return *(const f16x8 *)(A + ((2 * step + term) * MF_MB + mb) * 1024);
                    };
                    // the scales of this lane's rows, 16 mb + 4 grp ..
                    auto sa = [&](int mb) __attribute__((always_inline)) { return *(const f32x4 *)(meta_sa + 16 * mb + 4 * grp); };
                    buf ^= 1;
                    if (p == 0) stg.load(w, grp);
                    if constexpr (SF::MIN) if (p == KST / KA) {
                        // K positions 0..7 the sums' hi, 8..23 what is below it (times LO), then zeros
                        f16x8 fm, fs;
                        float d, dm;
                        stg.template sums_codes<SF::C>(w, grp == 0 ? 1.f : 1.f / LO, fm, fs);
                        stg.scales(w, d, dm);
#pragma unroll
                        for (int mb = 0; mb < MBS; mb++) {
                            const f16x8 sums = av(0, 0, mb);
                            const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(sums, fm, f32x4{0, 0, 0, 0}, 0, 0, 0), s = sa(mb);
                            acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(sums, fs, acc[mb], 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                tot[mb][i] = fmaf(fmaf(c[i], dm, fmaf(low[mb][i], 1.f / LO, acc[mb][i]) * d), s[i], tot[mb][i]);
                        }
                        continue;
                    }
#pragma unroll
                    for (int q = 0; q < KA; q++) {
                        const int kk = KA * p + q;
                        if (SF::SBK == 32 && kk >= nk) break;
                        uint4 f[SF::NF];
                        const float sd = SF::make(w, stg, kk, grp, f);
#pragma unroll
                        for (int mb = 0; mb < MBS; mb++) {
                            const f16x8 hi = av(q, 0, mb), lo = av(q, 1, mb);
                            const f32x4 z = {0, 0, 0, 0};
                            f32x4 c = SF::STEP || kk == 0 ? z : acc[mb], l = SF::STEP || kk == 0 ? z : low[mb];
                            l = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, as_f16x8(f[0]), l, 0, 0, 0);
                            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, as_f16x8(f[0]), c, 0, 0, 0);
                            if constexpr (SF::NF > 1) l = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, as_f16x8(f[1]), l, 0, 0, 0);
                            if constexpr (SF::STEP) {
#pragma unroll
                                for (int i = 0; i < 4; i++) acc[mb][i] = fmaf(fmaf(l[i], 1.f / LO, c[i]), sd, kk == 0 ? 0.f : acc[mb][i]);
                            } else {
                                acc[mb] = c;
                                low[mb] = l;
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);  // (the steps interleaved run out of registers)
                    }
                    if constexpr (!SF::MIN) if (p == KST / KA - 1) {
                        const float d = SF::scale(w);
#pragma unroll
                        for (int mb = 0; mb < MBS; mb++) {
                            const f32x4 s = sa(mb);
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                if constexpr (SF::STEP) tot[mb][i] = fmaf(acc[mb][i], s[i], tot[mb][i]);
                                else tot[mb][i] = fmaf(fmaf(low[mb][i], 1.f / LO, acc[mb][i]) * s[i], d, tot[mb][i]);
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        switch (mbs) {
        case 1: run_stages(Ic<1>{}); break;
        case 2: run_stages(Ic<2>{}); break;
        case 3: run_stages(Ic<3>{}); break;
        case 4: run_stages(Ic<4>{}); break;
        default: run_stages(Ic<5>{}); break;
        }

        // epilogue: lane holds picks 16 mb + 4 grp + i of weight row n
        const int n = nblk * S::RPB + wrow + l16;
        if constexpr (MODE == 0) {
            // half of the values each way between the gate and the up wave of the same rows, as in k_gmm
            float *xv = (float *)As;
            __syncthreads();
#pragma unroll
            for (int mb = 0; mb < MF_MB; mb++) {
                if (mb >= mbs) break;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int r = 16 * mb + 4 * grp + (mw == 0 ? 2 : 0) + i;
                    xv[r * S::RPB + wrow + l16] = mw == 0 ? tot[mb][2 + i] : tot[mb][i];
                }
            }
            __syncthreads();
            if (n < a.n) {
#pragma unroll
                for (int mb = 0; mb < MF_MB; mb++) {
                    if (mb >= mbs) break;
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int r = 16 * mb + 4 * grp + (mw == 0 ? 0 : 2) + i;
                        if (r >= tile.m) continue;
                        const float own = mw == 0 ? tot[mb][i] : tot[mb][2 + i], other = xv[r * S::RPB + wrow + l16];
                        float g = mw == 0 ? own : other, u = mw == 0 ? other : own, o;
                        if (a.act == CW_ACT_SILU) {
                            o = g / (1.0f + expf(-g)) * u;
                        } else {
                            const int64_t e = tile.expert;
                            if (a.bias0) g += a.bias0[e * a.n + n];
                            if (a.bias1) u += a.bias1[e * a.n + n];
                            g = fminf(g, a.limit);
                            u = fminf(fmaxf(u, -a.limit), a.limit);
                            o = (u + 1.0f) * (g * (1.0f / (1.0f + expf(-(g * a.alpha)))));
                        }
                        a.h[(int64_t)(tile.pos0 + r) * a.ldh + n] = o;
                    }
                }
            }
        } else {
            const bool split = MODE == 2 && a.split_cnt;
#pragma unroll
            for (int mb = 0; mb < MF_MB; mb++) {
                if (mb >= mbs) break;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int r = 16 * mb + 4 * grp + i;
                    if (r >= tile.m || n >= a.n) continue;
                    float *p = a.dn + blockIdx.y * a.split_stride + (int64_t)meta_pick[r] * a.n + n;
                    const float v = tot[mb][i];
                    if (split) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // at the coherence point
                    else *p = v;
                }
            }
            if (split) split_sum<S::RPB, S::NT>(a, item, nblk, tile.m, meta_pick, tid, &split_last);
        }
    }
}

// ------------------------------------------------------------------------------ pack

// One wave per NV * 256 values (blockIdx.y) of a row: hi and lo (times LO) of every value under a power of two per 256
// that brings their largest into [2^14, 2^15) (ascale: its inverse, one per 256), then, with SUMS, 32 halves
// per super-block: the 8 sub-block sums over 32 as hi, as two terms below it (times LO; together exact) and
// 8 zeros. 256 values that hold an infinity go in as +-2^14 for the infinities and 0 for the rest under an
// infinite ascale: every product then has the infinity's sign, or is a NaN where the weight is 0, as in f32
// (a NaN stays one).
template <int NV, bool SUMS>
__global__ __launch_bounds__(256) void k_pack_split(const float *x, int rows, int k, int ldx, uint16_t *a16, int lda, float *ascale,
                                                    PackExtra e) {
    if (blockIdx.y == 0) pack_extra(e);
    const int n_sb = (k + 255) / 256, row = blockIdx.x * 4 + (threadIdx.x >> 6), sb0 = NV * blockIdx.y, lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float *xr = x + (int64_t)row * ldx;
    float4 v[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = *(const float4 *)(xr + min(4 * lane + 256 * (sb0 + i), k - 4));
    uint16_t *o = a16 + (int64_t)row * lda;
    auto half = [](float f) -> uint32_t { return __builtin_bit_cast(uint16_t, (_Float16)f); };
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int sb = sb0 + i, c = 4 * lane + 256 * sb;
        if (sb >= n_sb) break;
        float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
        for (int q = 0; q < 4; q++) f[q] = c < k ? f[q] : 0.f;
        const float m = wave_max(fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3]))));
        float inv = INFINITY;
        if (m < INFINITY) {
            int ex = 0;
            if (m > 0.f) {
                frexpf(m, &ex);
                ex = min(15 - ex, 126);  // (values below 2^-111 keep a finite scale)
            }
            const float sc = ldexpf(1.0f, ex);
#pragma unroll
            for (int q = 0; q < 4; q++) f[q] *= sc;
            inv = ldexpf(1.0f, -ex);
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) f[q] = fabsf(f[q]) < INFINITY ? 0.f : f[q] == f[q] ? copysignf(16384.f, f[q]) : f[q];
        }
        if (lane == 0) ascale[(int64_t)row * n_sb + sb] = inv;
        if (c < k) {
            uint32_t h[4], l[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                h[q] = half(f[q]);
                l[q] = half((f[q] - (float)(_Float16)f[q]) * LO);
            }
            *(uint2 *)(o + c) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            *(uint2 *)(o + k + c) = make_uint2(l[0] | l[1] << 16, l[2] | l[3] << 16);
        }
        if constexpr (SUMS) {
            // in f64: through the codes' centre the sums carry the part that all weights of a sub-block share
            double s = ((double)f[0] + f[1]) + ((double)f[2] + f[3]);
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) s += __shfl_xor(s, d);
            s *= 1.0 / 32;
            const float h = (float)(_Float16)(float)s, r = (float)((s - h) * LO), l = (float)(_Float16)r;
            const uint32_t t[4] = {half(h), half(l), half((float)((s - h) * LO - l)), 0u};
            if ((lane & 7) < 4) o[2 * k + 32 * sb + 8 * (lane & 7) + (lane >> 3)] = (uint16_t)((lane & 2) ? (lane & 1) ? t[3] : t[2] : (lane & 1) ? t[1] : t[0]);
        }
    }
}

// ------------------------------------------------------------------------------ launchers

bool split_supported(int dtype) {
    return dtype == CW_Q4_K || dtype == CW_Q5_K || dtype == CW_Q6_K || dtype == CW_Q8_0;
}
static bool has_min(int dtype) { return dtype == CW_Q4_K || dtype == CW_Q5_K; }
// halves of a packed row (a multiple of 8: rows start on 16 bytes)
int split_row(int dtype, int64_t k) { return (int)(2 * k + (has_min(dtype) ? k / 256 * 32 : 0)); }
int split_scales(int64_t k) { return (int)((k + 255) / 256); }

int pack_rows_split(int dtype, const float *x, int rows, int k, int ldx, uint16_t *a16, float *ascale, hipStream_t s,
                    const PackExtra *extra) {
    if (rows == 0) return CW_OK;
    if (k % 32 || ldx % 4) return set_error(CW_ENOTSUP, "pack: row of %d (stride %d) is not whole K-steps", k, ldx);
    if (k > 8192) return set_error(CW_ENOTSUP, "pack: rows of %d above 8192", k);
    // two super-blocks per wave, four where the rows fill the device with those
    const int lda = split_row(dtype, k), n_sb = split_scales(k), nv = (int64_t)rows * n_sb >= 16384 ? 4 : 2;
    const dim3 grid((unsigned)((rows + 3) / 4), (unsigned)((n_sb + nv - 1) / nv)), block(256);
    const PackExtra e = extra ? *extra : PackExtra{};
#define CW_PACK(N, S) hipLaunchKernelGGL((k_pack_split<N, S>), grid, block, 0, s, x, rows, k, ldx, a16, lda, ascale, e)
    const bool sums = has_min(dtype);
    if (nv == 2 && sums) CW_PACK(2, true);
    else if (nv == 2) CW_PACK(2, false);
    else if (sums) CW_PACK(4, true);
    else CW_PACK(4, false);
#undef CW_PACK
    return check_launch("k_pack_split");
}

template <class SF, int MODE>
static int launch(const MfArgs &a, int tiles_max, int splits, hipStream_t s) {
    using S = SpShape<SF, MODE>;
    if (a.k % SF::SBK) return set_error(CW_ENOTSUP, "mfma: k %d is not a multiple of %d", a.k, SF::SBK);
    if ((int64_t)a.n * a.row_bytes > ((int64_t)1 << 32) - 16)  // (32-bit offsets from the 16-byte boundary below the matrix)
        return set_error(CW_ENOTSUP, "mfma: a matrix of %d rows of %lld bytes is 4 GiB or more", a.n, (long long)a.row_bytes);
    MfArgs b = a;
    int64_t items;
    b.run_tiles = run_of_tiles(tiles_max);
    if ((items = gemm_items(tiles_max, S::RPB, a.n)) >= ((int64_t)1 << 31)) return set_error(CW_ENOTSUP, "mfma: %lld work items", (long long)items);
    b.n_items = (int)items;
    const int64_t res = resident_blocks(S::PER_CU), blocks = items < res ? (items + 7) / 8 * 8 : res;
    static std::atomic<bool> lds_set[MAX_DEVICES];
    const int dev = current_device();
    if (!lds_set[dev].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute((const void *)k_gms<SF, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds_bytes()) != hipSuccess)
            return set_error(CW_EHIP, "mfma: cannot reserve %zu bytes of LDS", S::lds_bytes());
        lds_set[dev].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((k_gms<SF, MODE>), dim3((unsigned)blocks, (unsigned)splits), dim3(S::NT), S::lds_bytes(), s, b);
    return check_launch("k_gms");
}
template <int MODE>
static int by_fmt(int dtype, const MfArgs &a, int tiles_max, int splits, hipStream_t s) {
    if constexpr (MODE != 2) {  // (dense Q4_K and Q8_0 have the fp16 GEMM)
        if (dtype == CW_Q4_K) return launch<SQ4_K, MODE>(a, tiles_max, splits, s);
        if (dtype == CW_Q8_0) return launch<SQ8_0, MODE>(a, tiles_max, splits, s);
    }
    switch (dtype) {
    case CW_Q5_K: return launch<SQ5_K, MODE>(a, tiles_max, splits, s);
    case CW_Q6_K: return launch<SQ6_K, MODE>(a, tiles_max, splits, s);
    default: return set_error(CW_ENOTSUP, "mfma: dtype %d has no split-activation path", dtype);
    }
}
int split_gateup(int dtype, const MfArgs &a, int tiles_max, hipStream_t s) { return by_fmt<0>(dtype, a, tiles_max, 1, s); }
int split_down(int dtype, const MfArgs &a, int tiles_max, hipStream_t s) { return by_fmt<1>(dtype, a, tiles_max, 1, s); }

static size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }
constexpr int RPB2 = SpShape<SQ6_K, 2>::RPB, PER_CU2 = SpShape<SQ6_K, 2>::PER_CU;
size_t split_dense_workspace(int dtype, int64_t m, int64_t n, int64_t k) {
    int split_st;
    const int S = dense_splits(RPB2, 8, PER_CU2, m, n, k, split_st), tiles = (int)((m + MF_MT - 1) / MF_MT);
    return al256((size_t)m * split_row(dtype, k) * 2) + al256((size_t)m * split_scales(k) * 4) + al256(tiles * sizeof(MfTile)) + al256(4) +
           (S > 1 ? al256((size_t)S * m * n * 4) + al256((size_t)gemm_items(tiles, RPB2, n) * 4) : 0);
}
int split_dense(int dtype, const uint8_t *w, int64_t row_bytes, int n, int k, const float *x, int m, float *y, void *ws, size_t ws_bytes,
                hipStream_t s) {
    const size_t need = split_dense_workspace(dtype, m, n, k);
    if (ws_bytes < need || !ws) return set_error(CW_EINVAL, "qmatmul: workspace of %zu bytes, %zu needed", ws_bytes, need);
    int split_st;
    const int S = dense_splits(RPB2, 8, PER_CU2, m, n, k, split_st), tiles_n = (m + MF_MT - 1) / MF_MT;
    uint8_t *p = (uint8_t *)ws;
    uint16_t *x16 = (uint16_t *)p; p += al256((size_t)m * split_row(dtype, k) * 2);
    float *xs = (float *)p; p += al256((size_t)m * split_scales(k) * 4);
    MfTile *tiles = (MfTile *)p; p += al256((size_t)tiles_n * sizeof(MfTile));
    int *n_tiles = (int *)p; p += al256(4);
    float *part = nullptr;
    int *cnt = nullptr;
    if (S > 1) {
        part = (float *)p;
        p += al256((size_t)S * m * n * 4);
        cnt = (int *)p;
    }
    const PackExtra extra = {tiles, n_tiles, m, cnt, S > 1 ? (int)gemm_items(tiles_n, RPB2, n) : 0};
    int rc;
    if ((rc = pack_rows_split(dtype, x, m, k, k, x16, xs, s, &extra))) return rc;
    MfArgs a = {};
    a.w0 = w;
    a.row_bytes = row_bytes;
    a.n = n;
    a.k = k;
    a.a16 = x16;
    a.ascale = xs;
    a.lda = split_row(dtype, k);
    a.tiles = tiles;
    a.n_tiles = n_tiles;
    a.K = 1;
    a.dn = S > 1 ? part : y;
    a.split_st = S > 1 ? split_st : 0;
    a.split_stride = (int64_t)m * n;
    a.split_cnt = cnt;
    a.y = y;
    return by_fmt<2>(dtype, a, tiles_n, S, s);
}

}  // namespace cw
