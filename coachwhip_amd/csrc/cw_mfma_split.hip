// Grouped and dense GEMMs at f32 accuracy on the fp16 matrix instruction (gfx950), for the formats whose
// other path is one f32 matvec per row of x: Q5_K and Q6_K, and the formats they share a layer with.
//
// Every activation goes in as two fp16 terms of one power-of-two row scale, hi = fp16(x) and lo =
// fp16(x - hi), which together hold x to 2^-23 of itself (terms below 2^-24 of fp16's unit, 2^-39 of the
// row's largest value, vanish). The weight codes are integers that fp16 holds exactly: sc * q of Q4_K
// (at most 945) and Q5_K (at most 1,953), Q8_0's quants; Q6_K's sc * (q - 32) reaches
// 4,096 and goes in as its fp16 rounding and the exact rest (0 or +-1). A product then is two matrix
// instructions per fragment (three for Q6_K, whose rest times lo is below 2^-23 of the product), each
// product exact in the f32 accumulators. The minimum term of Q4_K and Q5_K is a ninth K-step per
// super-block: codes m against the sub-blocks' sums of x (computed in f32 by the pack, two fp16 terms).
// A super-block's sum is scaled into a second accumulator set in f32, so no running scale's rounding is
// carried through a row.
#include <math.h>

#include <atomic>

#include "cw_common.h"
#include "cw_gmm_dev.h"
#include "cw_mfma.h"
#include "cw_wave.h"

namespace cw {

// ------------------------------------------------------------------------------ formats
// Per format: NF code fragments per K-step of 32 weights (lane group grp: weights 8 grp .. 8 grp + 7),
// MIN the minimum step, STEP a scale per K-step instead of one per super-block (stage). Stage holds
// what a lane needs of its row for the whole stage; w is the row's window from the stage's first byte.

__device__ __forceinline__ uint4 codes_exact(uint32_t q0, uint32_t q1, float sc) {  // sc * q, q < 64
    return fma4(bytes_plus_1024(q0, q1), splat_f16f(sc), splat_f16f(-1024.0f * sc));
}
// scale and minimum of sub-block j from the 12 scale bytes of a Q4_K or Q5_K super-block (j a constant)
__device__ __forceinline__ void k4_const(const uint32_t (&b)[3], int j, uint32_t &sc, uint32_t &m) {
    const int sh = 8 * (j & 3);
    if (j < 4) {
        sc = (b[0] >> sh) & 63;
        m = (b[1] >> sh) & 63;
    } else {
        sc = ((b[2] >> sh) & 0xF) | (((b[0] >> (sh + 6)) & 3) << 4);
        m = ((b[2] >> (sh + 4)) & 0xF) | (((b[1] >> (sh + 6)) & 3) << 4);
    }
}
__device__ __forceinline__ uint4 k4_mins(const uint32_t (&b)[3]) {  // the 8 minima as fp16
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t s, m0, m1;
        k4_const(b, 2 * i, s, m0);
        k4_const(b, 2 * i + 1, s, m1);
        o[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz((float)m0, (float)m1));
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

struct SQ4_K {
    static constexpr int TS = 144, SBK = 256, NF = 1;
    static constexpr bool MIN = true, STEP = false;
    struct Stage {
        uint32_t b[3];
        float d, dm;
        __device__ __forceinline__ void load(const WinRef &w, int) {
            const uint32_t dd = w.u32(0);
            const uint2 lo = w.u64(4);
            b[0] = lo.x;
            b[1] = lo.y;
            b[2] = w.u32(12);
            d = h2f(dd & 0xFFFFu);
            dm = h2f(dd >> 16);
        }
        __device__ __forceinline__ uint4 mins() const { return k4_mins(b); }
    };
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &st, int kk, int grp, uint4 (&f)[1]) {
        uint32_t sc, m;
        k4_const(st.b, kk, sc, m);
        const uint2 q = w.u64(16 + 32 * (kk >> 1) + 8 * grp);
        const int sh = 4 * (kk & 1);
        f[0] = codes_exact((q.x >> sh) & 0x0F0F0F0Fu, (q.y >> sh) & 0x0F0F0F0Fu, (float)sc);
        return 0.f;
    }
};

struct SQ5_K {
    static constexpr int TS = 176, SBK = 256, NF = 1;
    static constexpr bool MIN = true, STEP = false;
    struct Stage {
        uint32_t b[3];
        uint2 h;  // the lane's bytes of qh: bit kk is weight kk's fifth
        float d, dm;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            const uint32_t dd = w.u32(0);
            const uint2 lo = w.u64(4);
            b[0] = lo.x;
            b[1] = lo.y;
            b[2] = w.u32(12);
            h = w.u64(16 + 8 * grp);
            d = h2f(dd & 0xFFFFu);
            dm = h2f(dd >> 16);
        }
        __device__ __forceinline__ uint4 mins() const { return k4_mins(b); }
    };
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &st, int kk, int grp, uint4 (&f)[1]) {
        uint32_t sc, m;
        k4_const(st.b, kk, sc, m);
        const uint2 q = w.u64(48 + 32 * (kk >> 1) + 8 * grp);
        const int sh = 4 * (kk & 1);
        f[0] = codes_exact(((q.x >> sh) & 0x0F0F0F0Fu) | (((st.h.x >> kk) & 0x01010101u) << 4),
                           ((q.y >> sh) & 0x0F0F0F0Fu) | (((st.h.y >> kk) & 0x01010101u) << 4), (float)sc);
        return 0.f;
    }
};

struct SQ6_K {
    static constexpr int TS = 210, SBK = 256, NF = 2;
    static constexpr bool MIN = false, STEP = false;
    struct Stage {
        uint32_t sc[4];  // the lane's half of each K-step: at bit 16 (kk & 1) of sc[kk >> 1]
        float d, dm;
        __device__ __forceinline__ void load(const WinRef &w, int grp) {
            const uint2 a = w.u64(192), b = w.u64(200);
            const int sh = 8 * (grp >> 1);
            sc[0] = a.x >> sh;
            sc[1] = a.y >> sh;
            sc[2] = b.x >> sh;
            sc[3] = b.y >> sh;
            d = h2f(w.u32(208) & 0xFFFFu);
        }
        __device__ __forceinline__ uint4 mins() const { return make_uint4(0, 0, 0, 0); }
    };
    static __device__ __forceinline__ float make(const WinRef &w, const Stage &st, int kk, int grp, uint4 (&f)[2]) {
        const int h = kk >> 2, r = kk & 3;
        const uint2 l = w.u64(64 * h + 32 * (r & 1) + 8 * grp), g = w.u64(128 + 32 * h + 8 * grp);
        const int sh = 4 * (r >> 1);
        const uint32_t q0 = ((l.x >> sh) & 0x0F0F0F0Fu) | (((g.x >> (2 * r)) & 0x03030303u) << 4);
        const uint32_t q1 = ((l.y >> sh) & 0x0F0F0F0Fu) | (((g.y >> (2 * r)) & 0x03030303u) << 4);
        const uint32_t sc = splat_f16f((float)(int8_t)(st.sc[kk >> 1] >> (16 * (kk & 1))));
        const uint4 c = fma4(bytes_plus_1024(q0, q1), 0x3C003C00u, 0xE420E420u);  // 1.0, -1056.0: q - 32
        f[0] = scale4(c, sc);
        // the rest of the product: c sc - fp16(c sc), exact
        const uint4 n = make_uint4(f[0].x ^ 0x80008000u, f[0].y ^ 0x80008000u, f[0].z ^ 0x80008000u, f[0].w ^ 0x80008000u);
        f[1] = make_uint4(pk_fma_u(c.x, sc, n.x), pk_fma_u(c.y, sc, n.y), pk_fma_u(c.z, sc, n.z), pk_fma_u(c.w, sc, n.w));
        return 0.f;
    }
};

struct SQ8_0 {
    static constexpr int TS = 34, SBK = 32, NF = 1;
    static constexpr bool MIN = false, STEP = true;
    struct Stage {
        float d, dm;
        __device__ __forceinline__ void load(const WinRef &, int) {}
        __device__ __forceinline__ uint4 mins() const { return make_uint4(0, 0, 0, 0); }
    };
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
// buffer a stage starts with a round trip to memory, and that is what bounds it. Against a matvec per row
// or pick: Q6_K 4001 x 4096 at 77 rows 215 -> 33 us (pack included), error against f64 2.1e-7 -> 1.7e-7; a
// layer of 128 experts, top-8, Q4_K 768 x 2048 and Q6_K 2048 x 768 at 301 tokens 2.3 ms -> about 0.25.
template <class SF, int MODE>
struct SpShape {
    static constexpr int KST = 8, NW = 8, NT = 64 * NW, NM = MODE == 0 ? 2 : 1, WPM = NW / NM, RPB = 16 * WPM;
    static constexpr int SEG = SF::SBK == 32 ? KST * SF::TS : SF::TS;
    static constexpr int PCS = ((SEG + 30) / 16) | 1, WB = 16 * PCS;  // pieces of a window (odd: LDS banks) and its bytes
    static constexpr int W_BYTES = NM * RPB * WB;
    static constexpr int KA = 2, PARTS = KST / KA + (SF::MIN ? 1 : 0);
    static constexpr int PART = KA * 2 * MF_MB * 1024, A_BYTES = 2 * PART;
    static constexpr int META = MF_MT * 8, PER_CU = 2;
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
    int *meta_pick = (int *)(meta_sa + MF_MT);
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
        if (tid < tile.m) {  // (the first stage's barriers publish these)
            const int pos = tile.pos0 + tid;
            meta_sa[tid] = a.ascale[a.rows ? a.rows[pos] : pos];
            meta_pick[tid] = a.pile_pick ? a.pile_pick[pos] : pos;
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
        const uint32_t as_lds = lds_addr(As), ws_lds = lds_addr(Ws);
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
                f32x4 acc[MBS];
#pragma unroll
                for (int p = 0; p < S::PARTS; p++) {
                    __builtin_amdgcn_s_waitcnt(0);  // this part's activations (and the windows)
                    __syncthreads();
                    if (p + 1 < S::PARTS) issue_a(st, p + 1, buf ^ 1);
                    else if (st + 1 < st_hi) issue_a(st + 1, 0, buf ^ 1);
                    const uint8_t *A = As + buf * S::PART + lane * 16;
                    auto av = [&](int step, int term, int mb) __attribute__((always_inline)) {
                        return *(const f16x8 *)(A + ((2 * step + term) * MF_MB + mb) * 1024);
                    };
                    buf ^= 1;
                    if (p == 0) stg.load(w, grp);
                    if (SF::MIN && p == KST / KA) {
                        const f16x8 m = as_f16x8(stg.mins());
                        const float sc = -32.f * stg.dm;  // (the sums are held over 32)
#pragma unroll
                        for (int mb = 0; mb < MBS; mb++) {
                            const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(av(0, 0, mb), m, f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 4; i++) tot[mb][i] = fmaf(c[i], sc, tot[mb][i]);
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
                            f32x4 c = SF::STEP || kk == 0 ? f32x4{0, 0, 0, 0} : acc[mb];
                            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, as_f16x8(f[0]), c, 0, 0, 0);
                            if constexpr (SF::NF > 1) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, as_f16x8(f[1]), c, 0, 0, 0);
                            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, as_f16x8(f[0]), c, 0, 0, 0);
                            acc[mb] = c;
                            if constexpr (SF::STEP) {
#pragma unroll
                                for (int i = 0; i < 4; i++) tot[mb][i] = fmaf(c[i], sd, tot[mb][i]);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);  // (the steps interleaved run out of registers)
                    }
                    if (!SF::STEP && p == KST / KA - 1) {
#pragma unroll
                        for (int mb = 0; mb < MBS; mb++)
#pragma unroll
                            for (int i = 0; i < 4; i++) tot[mb][i] = fmaf(acc[mb][i], stg.d, tot[mb][i]);
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
                    xv[r * S::RPB + wrow + l16] = (mw == 0 ? tot[mb][2 + i] : tot[mb][i]) * meta_sa[r];
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
                        const float own = (mw == 0 ? tot[mb][i] : tot[mb][2 + i]) * meta_sa[r], other = xv[r * S::RPB + wrow + l16];
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
                    const float v = tot[mb][i] * meta_sa[r];
                    if (split) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // at the coherence point
                    else *p = v;
                }
            }
            if (split) split_sum<S::RPB, S::NT>(a, item, nblk, tile.m, meta_pick, tid, &split_last);
        }
    }
}

// ------------------------------------------------------------------------------ pack

// One wave per row, as k_pack_f16: hi and lo of every value under the row's power-of-two scale (the
// largest value in [2^14, 2^15)), then, with SUMS, 32 halves per super-block: the 8 sub-block sums
// over 32 as hi, as lo, and 16 zeros.
template <int NV, bool SUMS>
__global__ __launch_bounds__(256) void k_pack_split(const float *x, int rows, int k, int ldx, uint16_t *a16, int lda, float *ascale,
                                                    PackExtra e) {
    pack_extra(e);
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float *xr = x + (int64_t)row * ldx;
    float4 v[NV];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = *(const float4 *)(xr + min(4 * lane + 256 * i, k - 4));
#pragma unroll
    for (int i = 0; i < NV; i++) {
        if (4 * lane + 256 * i >= k) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    }
    m = wave_max(m);
    int ex = 0;
    if (m > 0.f && m < INFINITY) {
        frexpf(m, &ex);
        ex = min(15 - ex, 126);  // (a row of values below 2^-111 keeps a finite scale)
    }
    const float sc = ldexpf(1.0f, ex);
    uint16_t *o = a16 + (int64_t)row * lda;
    auto hi_lo = [](float f, uint32_t &h, uint32_t &l) {
        const _Float16 a = (_Float16)f;
        const float rest = f - (float)a;
        h = __builtin_bit_cast(uint16_t, a);
        l = __builtin_bit_cast(uint16_t, (_Float16)(fabsf((float)a) < INFINITY ? rest : 0.f));  // an infinity (or NaN) has no rest
    };
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = 4 * lane + 256 * i;
        const float f[4] = {v[i].x * sc, v[i].y * sc, v[i].z * sc, v[i].w * sc};
        if (c < k) {
            uint32_t h[4], l[4];
#pragma unroll
            for (int q = 0; q < 4; q++) hi_lo(f[q], h[q], l[q]);
            *(uint2 *)(o + c) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            *(uint2 *)(o + k + c) = make_uint2(l[0] | l[1] << 16, l[2] | l[3] << 16);
        }
        if constexpr (SUMS) {
            const float s = group_sum<8>((f[0] + f[1]) + (f[2] + f[3])) * (1.0f / 32);
            uint32_t h, l;
            hi_lo(s, h, l);
            if (256 * i < k) {  // (whole super-blocks)
                uint16_t *so = o + 2 * k + 32 * i;
                if ((lane & 7) == 0) {
                    so[lane >> 3] = (uint16_t)h;
                    so[8 + (lane >> 3)] = (uint16_t)l;
                } else if ((lane & 7) <= 2) {
                    so[8 + 8 * (lane & 7) + (lane >> 3)] = 0;
                }
            }
        }
    }
    if (lane == 0) ascale[row] = ldexpf(1.0f, -ex);
}

// ------------------------------------------------------------------------------ launchers

bool split_supported(int dtype) {
    return dtype == CW_Q4_K || dtype == CW_Q5_K || dtype == CW_Q6_K || dtype == CW_Q8_0;
}
static bool has_min(int dtype) { return dtype == CW_Q4_K || dtype == CW_Q5_K; }
// halves of a packed row (a multiple of 8: rows start on 16 bytes)
int split_row(int dtype, int64_t k) { return (int)(2 * k + (has_min(dtype) ? k / 256 * 32 : 0)); }

int pack_rows_split(int dtype, const float *x, int rows, int k, int ldx, uint16_t *a16, float *ascale, hipStream_t s,
                    const PackExtra *extra) {
    if (rows == 0) return CW_OK;
    if (k % 32 || ldx % 4) return set_error(CW_ENOTSUP, "pack: row of %d (stride %d) is not whole K-steps", k, ldx);
    const dim3 grid((rows + 3) / 4);
    const int nv = (k + 255) / 256, lda = split_row(dtype, k);
    const PackExtra e = extra ? *extra : PackExtra{};
#define CW_PACK(N) \
    if (nv <= N) { \
        if (has_min(dtype)) hipLaunchKernelGGL((k_pack_split<N, true>), grid, dim3(256), 0, s, x, rows, k, ldx, a16, lda, ascale, e); \
        else hipLaunchKernelGGL((k_pack_split<N, false>), grid, dim3(256), 0, s, x, rows, k, ldx, a16, lda, ascale, e); \
        return check_launch("k_pack_split"); \
    }
    CW_PACK(2) CW_PACK(4) CW_PACK(8) CW_PACK(12) CW_PACK(16) CW_PACK(32)
#undef CW_PACK
    return set_error(CW_ENOTSUP, "pack: rows of %d above 8192", k);
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
    return al256((size_t)m * split_row(dtype, k) * 2) + al256(m * 4) + al256(tiles * sizeof(MfTile)) + al256(4) +
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
    float *xs = (float *)p; p += al256((size_t)m * 4);
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
