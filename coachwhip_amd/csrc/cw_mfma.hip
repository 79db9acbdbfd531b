// Grouped expert GEMMs on MFMA (gfx950, v_mfma_f32_16x16x32_f16) for the MoE layer's prefill.
//
// Picks are grouped by the slot they read (mfma_piles); a tile is up to MF_MT = 80 picks of one
// slot (5 MFMA blocks of 16) by RPB weight rows per matrix. A block has 8 waves (for gate/up, 4 on
// gate and 4 on up); each wave owns 16 weight rows and every pick block of the tile.
//
// Exactness: a weight is (f16 super-block scale) x (small integer code). The codes go through
// MFMA as fp16 integers, which they represent exactly: IQ2_XXS / IQ2_S codes (2s+1)*grid*sign
// are at most 31*43 = 1333, IQ3_XXS codes 8*(2s+1)*grid*sign multiples of 8 up to 8*31*62, IQ3_S
// codes (1+2s)*grid*sign at most 31*15 = 465, MXFP4 codes the doubled E2M1 values up to 12,
// IQ4_XS codes the non-linear levels (|v| <= 127, scaled per K-step like Q8_0). Products with fp16 activations are exact in the f32
// accumulators; the f32 scale of each super-block (d/8, d, or MXFP4's 2^(e-128) per 32) is
// applied to the partial sum of its K-steps. Activations are rounded to fp16 once, with a
// power-of-two scale per row (exact) so that no row overflows: that rounding (2^-11 relative)
// is the only approximation.
#include <atomic>
#include <type_traits>

#include "cw_common.h"
#include "cw_device.h"
#include "cw_gmm_dev.h"
#include "cw_mfma.h"
#include "cw_wave.h"

namespace cw {

// Tile shape of the grouped GEMM: a block owns one M-tile (up to MF_MT = 80 picks of a slot, in
// 16-row pick blocks) and RPB weight rows per matrix. Each wave takes NB blocks of 16 rows of one
// matrix and every pick block: per K-step it reads one activation fragment per pick block,
// decodes NB weight fragments and issues up to MF_MB*NB MFMAs. The decode is the VALU's work, so
// the LDS holds code tables that take work off the VALU, and the activations are shared by all
// waves of the block.
template <class MF, int MODE>
struct GmShape {
    static constexpr int LDS_MAX = 160 * 1024;
    static constexpr int NM = MODE == 0 ? 2 : 1;
    static constexpr int NB = 1;
    // PF: K-step table lookups and activation fragments read one step ahead (two register sets),
    // for every format but MXFP4 (equal or slower).
    static constexpr bool PF = !std::is_same<MF, MMXFP4>::value;
    // Blocks of 8 waves, two per CU, so one block's item start and end and its barriers' waits overlap
    // the other's K-steps. A wave works on one matrix (MODE 0: the first WPM waves on gate, the others on
    // up), which keeps its registers to one accumulator set.
    static constexpr int NW = 8, NT = 64 * NW, PER_CU = 2;
    static constexpr int WPM = NW / NM;                              // waves per matrix
    static constexpr int RPW = 16 * NB, RPB = WPM * RPW;
    static constexpr int W_BYTES = NM * RPB * Win<MF>::BYTES;       // one stage of weight windows
    static constexpr int META_BYTES = 2 * 128 * 4;                   // scale and pick of each row of the tile, by whole waves
    // The stage's activations load in HPS parts of KA K-steps, into a ring of as many parts of the tile's
    // pick blocks as the space of two full tiles holds; the windows into a ring of NWB stages. KA = 4
    // where three stages of windows fit beside it, else 2.
    static constexpr int a_bytes(int ka) { return 2 * ka * MF_MB * 64 * 16; }
    static constexpr int room(int ka) { return LDS_MAX / PER_CU - ((MF::LDS + 15) & ~15) - a_bytes(ka) - META_BYTES; }
    static constexpr int KA = room(4) >= 3 * W_BYTES ? 4 : 2;
    static constexpr int NWB = room(KA) >= 3 * W_BYTES ? 3 : 2;
    // MXFP4, whose K-steps are the shortest (a conversion per byte, no tables), feels the barrier per part
    // most: its ring takes what LDS the windows leave (less the kernel's static word, to whole KB), and tiles
    // of so few pick blocks that two parts of four K-steps fit (four, 64 rows) go in those. Dense 4096 x
    // 4096 at 16 rows 17.2 -> 16.5 us, 64 rows 25.5 -> 24.8, 80 rows (three parts of two) 28.6 -> 28.2, 8192 x
    // 1024 at 12 rows 12.1 -> 11.8; parts of eight at 32 rows and fewer measured the same.
    static constexpr bool WIDE = std::is_same<MF, MMXFP4>::value && KA == 2;
    static constexpr int A_BYTES = WIDE ? (room(0) - NWB * W_BYTES - 16) / 1024 * 1024 : a_bytes(KA);
    static constexpr int ka(int mbs) { return WIDE && 2 * 4 * mbs * 1024 <= A_BYTES ? 4 : KA; }
    static constexpr int hps(int mbs) { return MF::KST / ka(mbs); }
    // parts of the activation ring for MBS pick blocks: a part is requested NA - 1 parts ahead, and never
    // before the windows of its stage
    static constexpr int na(int mbs) {
        const int n = A_BYTES / (ka(mbs) * mbs * 1024), m = 1 + (NWB - 1) * hps(mbs);
        return n < m ? (n < 5 ? n : 5) : (m < 5 ? m : 5);
    }
    // Loads that may still be in flight when part hp of a stage starts: what its wave has requested after
    // the part's activations and, for the stage's first part, after the stage's windows (loads return in
    // order). HPS: parts per stage; ntw: a wave's window loads per stage; ka: its activation loads per part
    // (0 for the waves that load none).
    static constexpr int in_flight(int hp, int HPS, int NA, int ntw, int ka) {
        int n = ka * (NA - 2);
        for (int i = 1; i <= NA - 1; i++) n += (hp - i) % HPS == 0 ? ntw : 0;  // stage starts among the parts since
        if (hp == 0) {
            const int parts = (NWB - 1) * HPS - 1 < NA - 1 ? (NWB - 1) * HPS - 1 : NA - 1;
            const int w = ka * parts + ntw * (NWB - 2);
            if (w < n) n = w;
        }
        return n < 63 ? n : 63;
    }
    static constexpr int BASE_BYTES = ((MF::LDS + 15) & ~15) + A_BYTES + META_BYTES + NWB * W_BYTES;
    static constexpr size_t lds_bytes() { return BASE_BYTES; }
    static_assert(PER_CU * BASE_BYTES <= LDS_MAX, "the GEMM's LDS does not fit");
    static_assert(MODE != 0 || MF_MT * RPB * 4 <= A_BYTES, "the gate/up exchange does not fit the activation buffers");
};

// MODE 0: gate and up with the activation, hidden rows written in pile order.
// MODE 1: down, one output row per pick (combined per token by k_combine, in pick order, so the
//         result does not depend on the order blocks finish in).
// MODE 2: a dense matmul, the same output as MODE 1 (pile_pick NULL: one row per position).
//
// Per stage of 8 K-steps, the block copies its activations and the weight bytes of its rows
// into LDS with direct global-to-LDS loads: activations in MFMA fragment order ([K-step][pick
// block][lane] x 16 bytes, so every fragment read is one conflict-free ds_read_b128), weights as
// one window of whole 16-byte pieces per row (each load instruction covers 1 KB of consecutive
// pieces, instead of a few bytes from each of 16 rows). A piece is loaded only when it holds a byte of the row's stage; an aligned 16-byte
// piece cannot cross a page boundary, so its other bytes are mapped memory too.
//
// What bounds it: instructions. A wave's stage was about 300 VALU and 250 scalar instructions around 8
// fragments (half of them load addresses worked out in 64 bits, LDS addresses cast through a generic
// pointer, and M0 saved around every load); loads from a uniform base with 32-bit lane offsets, LDS
// addresses kept as such and rows that start on 16 bytes (Q4_K) taken as one constant make it about 230
// and 100 (IQ2_XXS gate/up of 1,500 tokens: 10.4 VALU and 4.0 scalar instructions per MFMA, three pick blocks
// a stage; 29 % of the waves' time issuing, 36 % on dependencies, 36 % at barriers and for loads, the matrix
// pipe 21 % busy). Longer prefetches alone (the rings below, before that) changed nothing. Two 8-wave blocks per
// CU for gate/up instead of one of 16 gave 8 % at 64 tokens. Layers, before and after all of it: 256 IQ2
// experts, top-8, 2048 x 512, 32 tokens 122 -> 106 us, 64 tokens 157 -> 137, 1,500 tokens 239 -> 230; 128
// Q4_K experts, 768 x 2048, 256 tokens 155 -> 145; 64 IQ4_XS experts, 16 tokens 121 -> 91; dense Q8_0 4096 x
// 4096, 512 rows 83 -> 65.
//
// Scales: the accumulator of a weight row carries a running scale. When a new scale unit starts
// (an IQ super-block, or an MXFP4 stage), the accumulator is multiplied by old/new scale and the
// unit's codes accumulate on top; the epilogue multiplies by the last scale. This keeps one
// accumulator per output instead of a partial sum per scale unit.
template <class MF, int MODE>
__global__ __launch_bounds__(1024, 4) void k_gmm(const MfArgs a) {
    using S = GmShape<MF, MODE>;
    using W = Win<MF>;
    constexpr int NB = S::NB, KST = MF::KST;
    constexpr int NM = 1;  // matrices per wave (a block has S::NM: gate/up waves are split)
    constexpr bool POW2 = MF::SCALE == 1, STEP = MF::SCALE == 2;
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int split_last;  // split-K: this block finished its work item's last split
    uint8_t *tab = smem;
    uint8_t *As = smem + ((MF::LDS + 15) & ~15);
    uint8_t *Ws = As + S::A_BYTES;
    float *meta_sa = (float *)(Ws + S::NWB * S::W_BYTES);
    int *meta_pick = (int *)(meta_sa + 128);
    const int n_nb = (a.n + S::RPB - 1) / S::RPB;
    // blocks go to the 8 XCDs round-robin; item b of each run of R*n_nb (R = run_tiles) takes
    // M-tile R*run + b%R and N-block b/R. With R = 8 an M-tile's N-blocks share an XCD (and its
    // L2 copy of the activations); with fewer tiles than 8, R < 8 spreads each tile's N-blocks
    // over R-strided XCDs instead of leaving XCDs idle.
    MF::fill(tab, threadIdx.x, S::NT);
    // Persistent blocks: block b takes work items b, b + gridDim.x, ... (gridDim.x is a multiple of
    // 8, so every item of a block maps to the block's XCD), and fills the code tables once.
    const int R = a.run_tiles, n_tiles = *a.n_tiles;
    for (int item = blockIdx.x; item < a.n_items; item += gridDim.x) {
        const int run = item / (R * n_nb), b = item - run * R * n_nb;
        const int mt = run * R + (b & (R - 1));
        if (mt >= n_tiles) continue;  // uniform across the block
        const int nblk = b / R;
        __syncthreads();  // the tables are in, and every wave is done with the previous item's LDS
        // lane values from an opaque copy of the thread index, so that nothing derived from them
        // is hoisted out of the item loop and kept in registers across items
        int tidi = threadIdx.x;
        asm("" : "+v"(tidi));
        const int tid = tidi, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = lane >> 4, l16 = lane & 15;
        const MfTile tile = a.tiles[mt];
        const int mbs = (tile.m + 15) >> 4;

        // The epilogue's activation scale and pick index of each tile row, by the first two waves straight
        // into LDS (rows past the tile's last: that one's, unused), published by the first part's barrier.
        const int mpos = tile.pos0 + min(tid, tile.m - 1);
        const int mrow = a.rows && wave < 2 ? a.rows[mpos] : mpos;

        // the activation row this lane copies: pick block `wave`, row l16, k-group grp
        const bool stager = wave < mbs;
        const int apos = tile.pos0 + min(16 * wave + l16, tile.m - 1);
        const uint16_t *asrc = a.a16 + (int64_t)(a.rows ? a.rows[apos] : apos) * a.lda + 8 * grp;

        if (wave < 2) {
            dma4(a.ascale + mrow, lds_addr(meta_sa) + 256 * wave);
            if (a.pile_pick) dma4(a.pile_pick + mpos, lds_addr(meta_pick) + 256 * wave);
            else meta_pick[tid] = mpos;
        }

        // Row r of the block is row nblk*RPB + r % RPB of matrix r / RPB (rows past n read the block's
        // first). Addresses are the first row of the block in its matrix (uniform) plus 32-bit offsets,
        // so they need no 64-bit registers per row.
        const int64_t row0 = (int64_t)nblk * S::RPB * a.row_bytes;
        const uint8_t *wb0 = a.w0 + (int64_t)tile.slot * a.s0 + row0;
        const uint8_t *wb1 = S::NM > 1 ? a.w1 + (int64_t)tile.slot * a.s1 + row0 : wb0;
        const int mw = S::NM > 1 ? wave / S::WPM : 0;  // this wave's matrix
        const int wrow = (wave - mw * S::WPM) * S::RPW;  // its first row within the matrix's N-block
        auto row_off = [&](int r, int m) -> uint32_t {  // byte offset of row r from the block's first of matrix m
            const int q = r - m * S::RPB;
            return (uint32_t)(nblk * S::RPB + q < a.n ? q : 0) * (uint32_t)a.row_bytes;
        };

        const int n_ks = a.k / 32, n_st = (n_ks + KST - 1) / KST;
        f32x4 acc[NM][NB][MF_MB];
        float rs[NM][NB];     // running scale (f16 scales) ...
        int rb[NM][NB];       // ... or running base exponent (MXFP4)
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int q = 0; q < NB; q++) {
                rs[m][q] = 1.f;
                rb[m][q] = 0;
#pragma unroll
                for (int mb = 0; mb < MF_MB; mb++) {
                    acc[m][q][mb] = f32x4{0, 0, 0, 0};
                    // the compiler must not treat the four elements as one value from here on: with
                    // that assumption it once fed later MFMAs three stale copies (wrong rows 1-3 of
                    // each 4-row group); the empty asm emits nothing
                    asm volatile("" : "+v"(acc[m][q][mb]));
                }
            }

        // The weight windows of stage st_w into buffer wbuf (an LDS address): every wave issues exactly NTW
        // loads (waves past the last piece repeat the first ones, writing the same bytes to the same
        // place, and pieces past a row's last one re-load that one into a slot nothing reads), so a
        // stage's wait can leave exactly the loads after it in flight. RPB*PCS is a multiple of 64: a
        // wave's pieces lie in one matrix and the matrix base stays scalar. A piece's row offset and its
        // place in the row's window are the same in every stage, so they are worked out once per tile
        // (the division by the window's piece count and the row's 32-bit multiply), from the 16-byte
        // boundary at or below the block's first row: wp_off the row's first byte, wp_p the piece.
        constexpr int NP = S::NM * S::RPB * W::PCS, NTW = (NP + S::NT - 1) / S::NT;
        static_assert(S::RPB * W::PCS % 64 == 0, "a wave's pieces lie in one matrix");
        const uint32_t b0 = (uint32_t)(uintptr_t)wb0 & 15, b1 = (uint32_t)(uintptr_t)wb1 & 15;
        const uint8_t *wa0 = wb0 - b0, *wa1 = wb1 - b1;
        constexpr bool ALIGNED = MF::TS % 16 == 0;  // every row starts at the base's place in its 16 bytes
        const uint32_t seg_all = MF::SBK == 32 ? (uint32_t)(MF::TS * KST) : (uint32_t)MF::TS;
        uint32_t wp_off[NTW], wp_p[NTW];
#pragma unroll
        for (int t = 0; t < NTW; t++) {
            const int w0 = S::NT * t + 64 * wave, i = (w0 < NP ? w0 : w0 - NP) + lane;
            const int r = i / W::PCS, m = S::NM > 1 ? __builtin_amdgcn_readfirstlane(r / S::RPB) : 0;
            wp_p[t] = (uint32_t)(i - r * W::PCS);
            wp_off[t] = row_off(r, m) + (m == 0 ? b0 : b1);
            if constexpr (ALIGNED) wp_off[t] = (wp_off[t] & ~15u) + 16 * min(wp_p[t], ((m == 0 ? b0 : b1) + seg_all - 1) >> 4);
        }
        auto issue_w = [&](int st_w, uint32_t wbuf) __attribute__((always_inline)) {
            const uint32_t seg_w = MF::SBK == 32 ? MF::TS * min(KST, n_ks - st_w * KST) : MF::TS;  // bytes of a row in this stage
            const uint32_t at = (uint32_t)(W::SEG * st_w);
#pragma unroll
            for (int t = 0; t < NTW; t++) {
                const int w0 = S::NT * t + 64 * wave, wi = w0 < NP ? w0 : w0 - NP;  // the wave's first piece
                const uint8_t *base = S::NM > 1 && wi >= S::RPB * W::PCS ? wa1 : wa0;
                uint32_t o = wp_off[t] + at;
                if constexpr (!ALIGNED) o = (o & ~15u) + 16 * min(wp_p[t], ((o & 15) + seg_w - 1) >> 4);
                dma16_s(base, o, wbuf + 16 * wi);
            }
        };
        // K-steps KA*p .. KA*p + KA-1 of the row (clamped to it where it may end in between: unused) into a
        // ring slot (an LDS address) of MBS pick blocks
        auto issue_a = [&](int p, uint32_t slot, auto mbs_c) __attribute__((always_inline)) {
            constexpr int MBS = decltype(mbs_c)::value, KA = S::ka(MBS);
            if (!stager) return;
#pragma unroll
            for (int kk = 0; kk < KA; kk++) {
                const int ks = p * KA + kk;
                dma16(asrc + (MF::SBK == 32 ? min(ks, n_ks - 1) : ks) * 32, slot + (kk * MBS + wave) * 1024);
            }
        };

        // this lane's rows: their start in global memory mod 16
        uint32_t lmis[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) lmis[q] = (mw == 0 ? b0 : b1) + (ALIGNED ? 0 : row_off(mw * S::RPB + wrow + 16 * q + l16, mw));

        const uint32_t as_lds = lds_addr(As), ws_lds = lds_addr(Ws);
        const int st_lo = a.split_st ? blockIdx.y * a.split_st : 0;
        const int st_hi = a.split_st ? min(n_st, st_lo + a.split_st) : n_st;
        // The stages, with the tile's count of 16-pick MFMA blocks as a constant. Pipeline: part p's
        // activations are requested at part p - (NA - 1), stage st's windows at the start of stage
        // st - (NWB - 1): a few hundred cycles of K-steps cover neither a round trip to L2 (the
        // activations) nor one to HBM. One barrier per part publishes its loads and frees the ring slots
        // that the loads issued after it overwrite. Near an item's end, where fewer loads are in flight
        // than in_flight counts on, a part waits for all of them.
        auto stages = [&](auto mbs_c) __attribute__((always_inline)) {
            constexpr int MBS = decltype(mbs_c)::value, KA = S::ka(MBS), HPS = S::hps(MBS), NA = S::na(MBS), SLOT = KA * MBS * 1024;
            const int p_lo = st_lo * HPS, p_hi = st_hi * HPS;
            // the loads before the first part, in the order that the parts before it would have issued them
#pragma unroll
            for (int q = 1 - NA < -(S::NWB - 1) * HPS ? 1 - NA : -(S::NWB - 1) * HPS; q < 0; q++) {
                if (q + NA - 1 >= 0 && p_lo + q + NA - 1 < p_hi) issue_a(p_lo + q + NA - 1, as_lds + (q + NA - 1) * SLOT, mbs_c);
                if (q % HPS == 0 && st_lo + q / HPS + S::NWB - 1 < st_hi)
                    issue_w(st_lo + q / HPS + S::NWB - 1, ws_lds + (q / HPS + S::NWB - 1) * S::W_BYTES);
            }
            int aslot = 0, wslot = 0;  // ring slots of the current part and stage
            for (int st = st_lo; st < st_hi; st++) {
                const int nk = min(KST, n_ks - st * KST);              // K-steps in this stage
                const int nke = MF::SBK == 32 ? nk : KST;              // super-block formats: every stage is whole
                uint8_t *const Wst = Ws + wslot * S::W_BYTES;
                // the start of part hp: its loads are in, the next ones go out
                const uint8_t *Ap;
                auto start_part = [&](auto hp_c) __attribute__((always_inline)) {
                    constexpr int hp = decltype(hp_c)::value;
                    const int p = st * HPS + hp;
                    const int last_w = (hp == 0 ? st - 1 : st) + S::NWB - 1;  // the last windows requested before this part
                    if (p + NA - 2 < p_hi && last_w < st_hi) {
                        constexpr int na = S::in_flight(hp, HPS, NA, NTW, KA), nb = S::in_flight(hp, HPS, NA, NTW, 0);
                        if (stager) __builtin_amdgcn_s_waitcnt((na & 15) | ((na >> 4) << 14) | (7 << 4) | (15 << 8));
                        else __builtin_amdgcn_s_waitcnt((nb & 15) | ((nb >> 4) << 14) | (7 << 4) | (15 << 8));
                    } else {
                        __builtin_amdgcn_s_waitcnt(0);
                    }
                    __syncthreads();
                    const int prev = aslot == 0 ? NA - 1 : aslot - 1;  // freed by the barrier
                    if (p + NA - 1 < p_hi) issue_a(p + NA - 1, as_lds + prev * SLOT, mbs_c);
                    if (hp == 0 && st + S::NWB - 1 < st_hi) issue_w(st + S::NWB - 1, ws_lds + (wslot == 0 ? S::NWB - 1 : wslot - 1) * S::W_BYTES);
                    Ap = As + aslot * SLOT;
                    aslot = aslot + 1 == NA ? 0 : aslot + 1;
                };
                start_part(Ic<0>{});

                // this lane's windows
                const uint8_t *win[NM][NB];
                WinRef wr[NM][NB];
                typename MF::Stage stg[NM][NB];
#pragma unroll
                for (int m = 0; m < NM; m++)
#pragma unroll
                    for (int q = 0; q < NB; q++) {
                        win[m][q] = Wst + (mw * S::RPB + wrow + 16 * q + l16) * W::BYTES + ((lmis[q] + (uint32_t)(W::SEG * st)) & 15);
                        wr[m][q] = WinRef::at<MF::ORG>(win[m][q]);
                        stg[m][q].load(wr[m][q], grp);
                    }

                bool zero[NM][NB];
                if constexpr (STEP) {
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int q = 0; q < NB; q++) zero[m][q] = false;
                } else if constexpr (POW2) {
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int q = 0; q < NB; q++) {
                            zero[m][q] = false;
                            // the base is the largest block exponent of the item's stages so far: the
                            // accumulators only ever move down onto a larger base (moving them up onto a
                            // smaller one overflowed f32 for rows whose block scales span more than 2^127)
                            int base = st > st_lo ? rb[m][q] : 0;
#pragma unroll
                            for (int kk = 0; kk < KST; kk++)
                                if (kk < nk) base = max(base, (int)MF::expo(win[m][q], kk));
                            if (st > st_lo && base != rb[m][q]) {
#pragma unroll
                                for (int mb = 0; mb < MBS; mb++)
#pragma unroll
                                    for (int i = 0; i < 4; i++) acc[m][q][mb][i] = ldexpf(acc[m][q][mb][i], rb[m][q] - base);
                            }
                            rb[m][q] = base;
                        }
                } else {
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int q = 0; q < NB; q++) {
                            // the accumulators move onto the new scale at the start of the K-steps (only
                            // the tile's pick blocks); a zero scale keeps the old one (its codes do not count)
                            const float d = stg[m][q].d;
                            zero[m][q] = d == 0.f;
                            const float ratio = d != 0.f ? rs[m][q] * __builtin_amdgcn_rcpf(d) : 1.f;
                            rs[m][q] = d != 0.f ? d : rs[m][q];
#pragma unroll
                            for (int mb = 0; mb < MBS; mb++) acc[m][q][mb] *= ratio;
                        }
                }

                // The K-steps, software pipelined so that no step waits on an LDS read it issued itself:
                // the window bytes of a step are requested two steps ahead, its table lookups and
                // activation fragments one step ahead (step kk issues those of kk+1 once its own fragment
                // is decoded, and they arrive while its MFMAs run). The first step of a part reads its
                // activations after the barrier that publishes them. A scheduling fence closes each step
                // (without it the compiler interleaves all eight steps and runs out of registers).
                typename MF::Raw rw[2][NM][NB];
                typename MF::Look lk[2][NM][NB];
                f16x8 av[2][MBS];
                auto issue_raw = [&](int kk) __attribute__((always_inline)) {
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int q = 0; q < NB; q++) rw[kk & 1][m][q] = MF::raw(wr[m][q], stg[m][q], kk, grp);
                };
                auto issue_look = [&](int kk) __attribute__((always_inline)) {
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int q = 0; q < NB; q++) lk[kk & 1][m][q] = MF::look(rw[kk & 1][m][q], stg[m][q], kk, grp, tab, zero[m][q]);
                };
                auto issue_av = [&](int kk) __attribute__((always_inline)) {
#pragma unroll
                    for (int mb = 0; mb < MBS; mb++) av[kk & 1][mb] = *(const f16x8 *)(Ap + (((kk % KA) * MBS + mb) * 64 + lane) * 16);
                };
                issue_raw(0);
                if (1 < nke) issue_raw(1);
                if constexpr (S::PF) {
                    issue_look(0);
                    issue_av(0);
                }
                auto step = [&](auto kk_c) __attribute__((always_inline)) {
                    constexpr int kk = decltype(kk_c)::value;
                    if (kk >= nke) return;  // uniform
                    if constexpr (kk > 0 && kk % KA == 0) {
                        start_part(Ic<kk / KA>{});
                        if constexpr (S::PF) issue_av(kk);
                    }
                    if constexpr (!S::PF) {
                        issue_look(kk);
                        issue_av(kk);
                    }
                    if constexpr (STEP) {
                        // a scale per K-step: move each accumulator onto it
#pragma unroll
                        for (int m = 0; m < NM; m++)
#pragma unroll
                            for (int q = 0; q < NB; q++) {
                                const float d = MF::step_scale(rw[kk & 1][m][q]);
                                zero[m][q] = d == 0.f;
                                if (d != 0.f) {
                                    const float ratio = __fdividef(rs[m][q], d);
#pragma unroll
                                    for (int mb = 0; mb < MBS; mb++) acc[m][q][mb] *= ratio;
                                    rs[m][q] = d;
                                }
                            }
                    }
                    f16x8 bf[NM][NB];
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int q = 0; q < NB; q++) {
                            if constexpr (POW2)
                                bf[m][q] = as_f16x8(MF::make_mx(rw[kk & 1][m][q], grp, (int)rw[kk & 1][m][q].e - rb[m][q]));
                            else
                                bf[m][q] = as_f16x8(MF::make(rw[kk & 1][m][q], lk[kk & 1][m][q], stg[m][q], kk, grp, zero[m][q]));
                        }
                    if (kk + 2 < KST && kk + 2 < nke) issue_raw(kk + 2);  // into the buffer step kk has just used
                    if (S::PF && kk + 1 < KST && kk + 1 < nke) {
                        issue_look(kk + 1);
                        if ((kk + 1) % KA != 0) issue_av(kk + 1);
                    }
#pragma unroll
                    for (int mb = 0; mb < MBS; mb++)
#pragma unroll
                        for (int m = 0; m < NM; m++)
#pragma unroll
                            for (int q = 0; q < NB; q++) {
                                acc[m][q][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[kk & 1][mb], bf[m][q], acc[m][q][mb], 0, 0, 0);
                            }
                    __builtin_amdgcn_sched_barrier(0);
                };
                step(Ic<0>{}); step(Ic<1>{}); step(Ic<2>{}); step(Ic<3>{});
                if constexpr (KST > 4) { step(Ic<4>{}); step(Ic<5>{}); step(Ic<6>{}); step(Ic<7>{}); }
                // a row's last stage may end before its later parts: their barriers all the same (they
                // were requested, and their slots count)
                if constexpr (MF::SBK == 32) {
                    if constexpr (HPS > 1) if (nke <= KA) start_part(Ic<1>{});
                    if constexpr (HPS > 2) if (nke <= 2 * KA) start_part(Ic<2>{});
                    if constexpr (HPS > 3) if (nke <= 3 * KA) start_part(Ic<3>{});
                }
                wslot = wslot + 1 == S::NWB ? 0 : wslot + 1;
            }
        };
        switch (mbs) {
        case 1: stages(Ic<1>{}); break;
        case 2: stages(Ic<2>{}); break;
        case 3: stages(Ic<3>{}); break;
        case 4: stages(Ic<4>{}); break;
        default: stages(Ic<5>{}); break;
        }

        // epilogue: lane holds picks 16*mb + 4*grp + i (i < 4) of weight row n (block q)
        float fs[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) fs[q] = POW2 ? ldexpf(1.0f, rb[0][q] - 128) : rs[0][q];
        if constexpr (MODE == 0) {
            // The gate wave and the up wave of the same rows hand each other half of their values through
            // LDS (the activation buffers, free once every wave is past the last K-step): the gate wave
            // finishes rows 4*grp and 4*grp + 1 of each pick block, the up wave the other two.
            float *xv = (float *)As;
            __syncthreads();
#pragma unroll
            for (int mb = 0; mb < MF_MB; mb++) {
                if (mb >= mbs) break;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int r = 16 * mb + 4 * grp + (mw == 0 ? 2 : 0) + i;
#pragma unroll
                    for (int q = 0; q < NB; q++) xv[r * S::RPB + wrow + 16 * q + l16] = (mw == 0 ? acc[0][q][mb][2 + i] : acc[0][q][mb][i]) * fs[q] * meta_sa[r];
                }
            }
            __syncthreads();
#pragma unroll
            for (int mb = 0; mb < MF_MB; mb++) {
                if (mb >= mbs) break;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int r = 16 * mb + 4 * grp + (mw == 0 ? 0 : 2) + i;
                    if (r >= tile.m) continue;
                    const int pos = tile.pos0 + r;
#pragma unroll
                    for (int q = 0; q < NB; q++) {
                        const int n = nblk * S::RPB + wrow + 16 * q + l16;
                        if (n >= a.n) continue;
                        const float own = (mw == 0 ? acc[0][q][mb][i] : acc[0][q][mb][2 + i]) * fs[q] * meta_sa[r];
                        const float other = xv[r * S::RPB + wrow + 16 * q + l16];
                        // sigmoid(z) = 1 / (1 + 2^(-z log2 e)) on the hardware's exp2 and
                        // reciprocal (each within 1 ulp)
                        constexpr float LOG2E = 1.4426950408889634f;
                        float g = mw == 0 ? own : other, u = mw == 0 ? other : own, o;
                        if (a.act == CW_ACT_SILU) {
                            o = g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * LOG2E)) * u;
                        } else {
                            const int64_t e = tile.expert;  // every pick of the tile's
                            if (a.bias0) g += a.bias0[e * a.n + n];
                            if (a.bias1) u += a.bias1[e * a.n + n];
                            g = fminf(g, a.limit);
                            u = fminf(fmaxf(u, -a.limit), a.limit);
                            o = (u + 1.0f) * (g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(g * a.alpha) * LOG2E)));
                        }
                        a.h[(int64_t)pos * a.ldh + n] = o;
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
                    if (r >= tile.m) continue;
                    const int pick = meta_pick[r];
#pragma unroll
                    for (int q = 0; q < NB; q++) {
                        const int n = nblk * S::RPB + wrow + 16 * q + l16;
                        if (n >= a.n) continue;
                        float *p = a.dn + blockIdx.y * a.split_stride + (int64_t)pick * a.n + n;
                        const float v = acc[0][q][mb][i] * fs[q] * meta_sa[r];
                        if (split)
                            __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // at the coherence point
                        else
                            *p = v;
                    }
                }
            }
            if (split) split_sum<S::RPB, S::NT>(a, item, nblk, tile.m, meta_pick, tid, &split_last);
        }
    }
}

// ------------------------------------------------------------------------------ helpers

// sum of the first n entries of a small LDS array
__device__ __forceinline__ int wc_total(const int *w, int n) {
    int t = 0;
    for (int i = 0; i < n; i++) t += w[i];
    return t;
}

// Inclusive prefix sum across the wave (six shuffle steps)
__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(v, d);
        if (lane >= d) v += u;
    }
    return v;
}

// One block: histogram of slots (or experts), exclusive scans, scatter of picks into their piles, tiles.
// Each thread reads its (up to) PILE_PER slots into registers before using any, so the loads
// overlap, and keeps them for the scatter; the order of picks inside a pile does not matter
// (every pick's outputs are computed independently of the other rows of its tile). Up to
// PILE_LDS picks, the scatter goes to LDS and the piles leave in coalesced stores (random 4-byte
// stores from one CU cost a memory transaction each).
// BY_EXPERT: a pile per expert (n_keys of them) instead of per slot: with a bias per expert, picks that
// share a slot but not an expert (experts that the bank does not hold all read slot 0) need tiles of their
// own.
constexpr int PILE_PER = 16, PILE_LDS = 12288;
template <bool BY_EXPERT>
__global__ __launch_bounds__(1024) void k_piles(const uint32_t *slots, const uint32_t *ids, int TK, int K, int n_slots, int n_keys,
                                                 int *pile_pick, int *pile_tok, MfTile *tiles, int *n_tiles) {
    __shared__ int cnt[1024], off[1024], cur[1024], rep[1024], wtot[16], wttot[16], wftot[16];
    __shared__ int staged[PILE_LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    cnt[tid] = 0;
    cur[tid] = 0;
    rep[tid] = 0;
    const bool one = TK <= 1024 * PILE_PER;  // the common case: every slot read once, kept in registers
    uint32_t v[PILE_PER];
    // the pile of pick i (none past the last one, or for a slot past the bank)
    auto key = [&](int i) __attribute__((always_inline)) -> uint32_t {
        if (i >= TK) return 0xFFFFFFFFu;
        if constexpr (BY_EXPERT) return slots[i] < (uint32_t)n_slots ? ids[i] : 0xFFFFFFFFu;
        else return slots[i];
    };
#pragma unroll
    for (int q = 0; q < PILE_PER; q++) v[q] = key(q * 1024 + tid);
    __syncthreads();
    for (int c0 = 0; c0 < TK; c0 += 1024 * PILE_PER) {
        if (c0) {
#pragma unroll
            for (int q = 0; q < PILE_PER; q++) v[q] = key(c0 + q * 1024 + tid);
        }
#pragma unroll
        for (int q = 0; q < PILE_PER; q++)
            if (v[q] < (uint32_t)n_keys) {
                atomicAdd(&cnt[v[q]], 1);
                atomicMax(&rep[v[q]], c0 + q * 1024 + tid);  // a pick of the slot, for its expert id
            }
    }
    __syncthreads();
    // exclusive scans of the counts, the tile counts and the first tiles: per wave, then over the
    // 16 wave totals. The tile list holds every slot's first tile, then the later tiles of the
    // slots with more than MF_MT picks: the GEMMs hand out work items in list order, so the last
    // round of items, which only some blocks run, takes the (smaller) remainder tiles.
    const int c = tid < n_keys ? cnt[tid] : 0;
    const int tc = (c + MF_MT - 1) / MF_MT, fc = c > 0 ? 1 : 0;
    const int ic = wave_incl_scan(c, lane), itc = wave_incl_scan(tc, lane), ifc = wave_incl_scan(fc, lane);
    if (lane == 63) {
        wtot[wave] = ic;
        wttot[wave] = itc;
        wftot[wave] = ifc;
    }
    __syncthreads();
    int wc = 0, wtc = 0, wfc = 0, nf = 0;
    for (int w = 0; w < 16; w++) {
        if (w < wave) {
            wc += wtot[w];
            wtc += wttot[w];
            wfc += wftot[w];
        }
        nf += wftot[w];
    }
    const int my_off = wc + ic - c, my_toff = wtc + itc - tc, my_f = wfc + ifc - fc;
    if (tid == 1023) *n_tiles = my_toff + tc;
    off[tid] = my_off;
    if (tid < n_keys) {
        const int ex = !BY_EXPERT && ids && c > 0 ? (int)ids[rep[tid]] : tid, sl = BY_EXPERT && c > 0 ? (int)slots[rep[tid]] : tid;
        for (int q = 0; q < tc; q++)
            tiles[q == 0 ? my_f : nf + (my_toff - my_f) + q - 1] = MfTile{sl, my_off + q * MF_MT, min(MF_MT, c - q * MF_MT), ex};
    }
    __syncthreads();
    for (int c0 = 0; c0 < TK; c0 += 1024 * PILE_PER) {
        if (!one) {
#pragma unroll
            for (int q = 0; q < PILE_PER; q++) v[q] = key(c0 + q * 1024 + tid);
        }
#pragma unroll
        for (int q = 0; q < PILE_PER; q++) {
            const int i = c0 + q * 1024 + tid;
            if (v[q] < (uint32_t)n_keys) {
                const int pos = off[v[q]] + atomicAdd(&cur[v[q]], 1);
                if (TK <= PILE_LDS) {
                    staged[pos] = i;
                } else {
                    pile_pick[pos] = i;
                    pile_tok[pos] = i / K;
                }
            }
        }
    }
    if (TK <= PILE_LDS) {
        __syncthreads();
        const int n = wtot[15] + wc_total(wtot, 15);  // picks that resolved to a slot
        for (int p = tid; p < n; p += 1024) {
            const int i = staged[p];
            pile_pick[p] = i;
            pile_tok[p] = i / K;
        }
    }
}

// One wave per row, the row held in registers (NV float4 per lane, k <= 256*NV): scale =
// 2^(15 - e) with max|x| in [2^(e-1), 2^e) keeps the row's largest value in [2^14, 2^15) of
// fp16 (below it for rows under 2^-111); ascale receives 1/scale.
template <int NV, int ORDER>
__global__ __launch_bounds__(256) void k_pack_f16(const float *x, int rows, int k, int ldx, uint16_t *a16, float *ascale,
                                                  PackExtra e) {
    pack_extra(e);
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float *xr = x + (int64_t)row * ldx;
    float4 v[NV];
    float m = 0.f;
    // loads from clamped addresses (all in flight at once), the values past the row zeroed after
    if constexpr (ORDER == K_PAIRS) {
        // positions c..c+3 of a 32-wide step take its elements 2t, 2t+16, 2t+1, 2t+17 (t = (c % 32) / 4)
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int c = min(4 * lane + 256 * i, k - 4);
            const float *b = xr + (c & ~31) + ((c & 31) >> 1);
            const float2 lo = *(const float2 *)b, hi = *(const float2 *)(b + 16);
            v[i] = make_float4(lo.x, hi.x, lo.y, hi.y);
        }
    } else {
#pragma unroll
        for (int i = 0; i < NV; i++) v[i] = *(const float4 *)(xr + min(4 * lane + 256 * i, k - 4));
    }
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (4 * lane + 256 * i >= k) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    }
    m = wave_max(m);
    int ex = 0;
    if (m > 0.f && m < INFINITY) {
        frexpf(m, &ex);
        ex = min(15 - ex, 126);  // (a row of values below 2^-111 keeps a finite scale, and 1 / scale stays normal)
    }
    const float sc = ldexpf(1.0f, ex);
    uint16_t *o = a16 + (int64_t)row * k;
    // K_OCTETS: the lane's 4 values are half (lane & 1) of octet l = (lane >> 1) & 3 of sub-block 4j + g =
    // lane >> 3: positions 32 (4j + l) + 8g
    const int c0 = ORDER == K_OCTETS ? 128 * (lane >> 5) + 32 * ((lane >> 1) & 3) + 8 * ((lane >> 3) & 3) + 4 * (lane & 1) : 4 * lane;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = c0 + 256 * i;
        if (c < k) {
            const uint32_t lo = __builtin_bit_cast(uint16_t, (_Float16)(v[i].x * sc)) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(v[i].y * sc)) << 16);
            const uint32_t hi = __builtin_bit_cast(uint16_t, (_Float16)(v[i].z * sc)) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(v[i].w * sc)) << 16);
            *(uint2 *)(o + c) = make_uint2(lo, hi);
        }
    }
    if (lane == 0) ascale[row] = ldexpf(1.0f, -ex);
}

// one thread per 4 outputs of a token: the weighted sum of its K picks' rows, bias added per pick,
// in pick order. A pick whose slot is out of range is in no pile and has no row: it contributes
// NaN, as it does on the matvec and decode paths. The picks go in chunks of CH, each chunk's
// slots, weights and expert ids loaded together, then its rows and bias rows (every pick has a
// row of dn, written or not, so those loads need no branch; past K a chunk reads pick K - 1
// again, unused).
template <int CH>
__global__ __launch_bounds__(256) void k_combine(const float *dn, const float *w, const float *bias, const uint32_t *ids,
                                                 const uint32_t *slots, uint32_t n_slots, int K, int H, float *out) {
    const int t = blockIdx.y, j = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (j >= H) return;
    const float nan = __int_as_float(0x7fc00000);
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int e0 = 0; e0 < K; e0 += CH) {
        uint32_t sl[CH], id[CH];
        float we[CH];
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int64_t pick = (int64_t)t * K + min(e0 + c, K - 1);
            sl[c] = slots[pick];
            we[c] = w[pick];
            id[c] = bias ? ids[pick] : 0u;
        }
        float4 d[CH], b[CH];
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int64_t pick = (int64_t)t * K + min(e0 + c, K - 1);
            d[c] = *(const float4 *)(dn + pick * H + j);
            b[c] = bias ? *(const float4 *)(bias + (int64_t)id[c] * H + j) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int c = 0; c < CH; c++) {
            if (e0 + c >= K) break;
            float4 v = sl[c] < n_slots ? d[c] : make_float4(nan, nan, nan, nan);
            if (bias) {
                v.x += b[c].x; v.y += b[c].y; v.z += b[c].z; v.w += b[c].w;
            }
            const float wc = we[c];
            acc.x += v.x * wc; acc.y += v.y * wc; acc.z += v.z * wc; acc.w += v.w * wc;
        }
    }
    *(float4 *)(out + (int64_t)t * H + j) = acc;
}

__global__ void k_fill_zero(float *p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0.f;
}

// ------------------------------------------------------------------------------ launchers

bool mfma_supported(int dtype) {
    return dtype == CW_IQ2_XXS || dtype == CW_IQ2_S || dtype == CW_IQ3_S || dtype == CW_MXFP4 || dtype == CW_Q4_K || dtype == CW_Q8_0 ||
           dtype == CW_Q2_K || dtype == CW_IQ3_XXS || dtype == CW_IQ4_XS || dtype == CW_MXFP4_R16;
}

int max_tiles(int TK, int n_piles) { return (TK + MF_MT - 1) / MF_MT + (n_piles < TK ? n_piles : TK); }

int mfma_piles(const uint32_t *slots, const uint32_t *ids, int TK, int K, int n_slots, int n_experts, int *pile_pick, int *pile_tok,
               MfTile *tiles, int *n_tiles, hipStream_t s) {
    if (n_slots > 1024 || n_experts > 1024) return set_error(CW_ENOTSUP, "mfma: %d slots, %d experts (1024 max)", n_slots, n_experts);
    if (n_experts) hipLaunchKernelGGL(k_piles<true>, dim3(1), dim3(1024), 0, s, slots, ids, TK, K, n_slots, n_experts, pile_pick, pile_tok, tiles, n_tiles);
    else hipLaunchKernelGGL(k_piles<false>, dim3(1), dim3(1024), 0, s, slots, ids, TK, K, n_slots, n_slots, pile_pick, pile_tok, tiles, n_tiles);
    return check_launch("k_piles");
}

int pack_rows_f16(const float *x, int rows, int k, int ldx, uint16_t *a16, float *ascale, hipStream_t s,
                  const PackExtra *extra, int order) {
    if (rows == 0) return CW_OK;
    if (k % 4 || ldx % 4) return set_error(CW_ENOTSUP, "pack: row of %d (stride %d) is not whole float4s", k, ldx);
    if (order != K_NATURAL && k % (order == K_OCTETS ? 256 : 32))
        return set_error(CW_ENOTSUP, "pack: a permuted row of %d is not whole steps", k);
    const dim3 grid((rows + 3) / 4);
    const int nv = (k + 255) / 256;
    const PackExtra e = extra ? *extra : PackExtra{};
#define CW_PACK(N) \
    if (nv <= N) { \
        if (order == K_PAIRS) hipLaunchKernelGGL((k_pack_f16<N, K_PAIRS>), grid, dim3(256), 0, s, x, rows, k, ldx, a16, ascale, e); \
        else if (order == K_OCTETS) hipLaunchKernelGGL((k_pack_f16<N, K_OCTETS>), grid, dim3(256), 0, s, x, rows, k, ldx, a16, ascale, e); \
        else hipLaunchKernelGGL((k_pack_f16<N, K_NATURAL>), grid, dim3(256), 0, s, x, rows, k, ldx, a16, ascale, e); \
        return check_launch("k_pack_f16"); \
    }
    CW_PACK(2) CW_PACK(4) CW_PACK(8) CW_PACK(12) CW_PACK(16) CW_PACK(32)
#undef CW_PACK
    return set_error(CW_ENOTSUP, "pack: rows of %d above 8192", k);
}

int combine_picks(const float *dn, const float *w, const float *bias, const uint32_t *ids, const uint32_t *slots, int n_slots,
                  int T, int K, int H, float *out, hipStream_t s) {
    if (T == 0) return CW_OK;
    if (H % 4) return set_error(CW_ENOTSUP, "combine: width %d is not a multiple of 4", H);
    const dim3 grid((H / 4 + 255) / 256, T);
    hipLaunchKernelGGL(k_combine<4>, grid, dim3(256), 0, s, dn, w, bias, ids, slots, (uint32_t)n_slots, K, H, out);
    return check_launch("k_combine");
}

int fill_zero(float *p, int64_t n, hipStream_t s) {
    if (n == 0) return CW_OK;
    int64_t b = (n + 255) / 256;
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)(b < 8192 ? b : 8192)), dim3(256), 0, s, p, n);
    return check_launch("k_fill_zero");
}

int run_of_tiles(int64_t tiles) { return tiles >= 8 ? 8 : tiles >= 4 ? 4 : tiles >= 2 ? 2 : 1; }
int64_t gemm_items(int64_t tiles, int rpb, int64_t n) {
    const int64_t R = run_of_tiles(tiles);
    return (tiles + R - 1) / R * R * ((n + rpb - 1) / rpb);
}

int current_device() {
    int dev = 0;
    return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < MAX_DEVICES ? dev : 0;
}

// persistent GEMM blocks: per_cu per CU of the current device, a multiple of 8 (the XCD count)
int64_t resident_blocks(int per_cu) {
    static std::atomic<int> cus_of[MAX_DEVICES];
    const int dev = current_device();
    int cus = cus_of[dev].load(std::memory_order_relaxed);
    if (!cus) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8) n = 256;
        cus = n / 8 * 8;
        cus_of[dev].store(cus, std::memory_order_relaxed);
    }
    return (int64_t)cus * per_cu;
}

template <class MF, int MODE>
static int launch(const MfArgs &a, int tiles_max, int splits, hipStream_t s) {
    using S = GmShape<MF, MODE>;
    if (a.k % MF::SBK) return set_error(CW_ENOTSUP, "mfma: k %d is not a multiple of %d", a.k, MF::SBK);
    if ((int64_t)a.n * a.row_bytes >= ((int64_t)1 << 32))
        return set_error(CW_ENOTSUP, "mfma: a matrix of %d rows of %lld bytes is 4 GiB or more", a.n, (long long)a.row_bytes);
    const int R = run_of_tiles(tiles_max);
    const int64_t items = gemm_items(tiles_max, S::RPB, a.n);
    if (items >= ((int64_t)1 << 31)) return set_error(CW_ENOTSUP, "mfma: %lld work items", (long long)items);
    const int64_t res = resident_blocks(S::PER_CU);
    const int64_t blocks = items < res ? (items + 7) / 8 * 8 : res;
    static std::atomic<bool> lds_set[MAX_DEVICES];  // dynamic LDS above 64 KB, opted into once per kernel and device
    const int dev = current_device();
    if (!lds_set[dev].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute((const void *)k_gmm<MF, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds_bytes()) != hipSuccess)
            return set_error(CW_EHIP, "mfma: cannot reserve %zu bytes of LDS", S::lds_bytes());
        lds_set[dev].store(true, std::memory_order_release);
    }
    MfArgs b = a;
    b.run_tiles = R;
    b.n_items = (int)items;
    hipLaunchKernelGGL((k_gmm<MF, MODE>), dim3((unsigned)blocks, (unsigned)splits), dim3(S::NT), S::lds_bytes(), s, b);
    return check_launch("k_gmm");
}

template <int MODE>
static int by_fmt(int dtype, const MfArgs &a, int tiles_max, int splits, hipStream_t s) {
    switch (dtype) {
    case CW_IQ2_XXS: return launch<MIQ2_XXS, MODE>(a, tiles_max, splits, s);
    case CW_IQ2_S: return launch<MIQ2_S, MODE>(a, tiles_max, splits, s);
    case CW_IQ3_S: return launch<MIQ3_S, MODE>(a, tiles_max, splits, s);
    case CW_MXFP4: return launch<MMXFP4, MODE>(a, tiles_max, splits, s);
    case CW_Q4_K: return launch<MQ4_K, MODE>(a, tiles_max, splits, s);
    case CW_Q8_0: return launch<MQ8_0, MODE>(a, tiles_max, splits, s);
    case CW_Q2_K: return launch<MQ2_K, MODE>(a, tiles_max, splits, s);
    case CW_IQ3_XXS: return launch<MIQ3_XXS, MODE>(a, tiles_max, splits, s);
    case CW_IQ4_XS: return launch<MIQ4_XS, MODE>(a, tiles_max, splits, s);
    default: return set_error(CW_ENOTSUP, "mfma: dtype %d has no MFMA path", dtype);
    }
}

static size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }

// the dense GEMM's N-block rows and stage size for a format (GmShape<MF, 2>)
template <class MF>
static void shape_of(int &rpb, int &kst, int &per_cu) {
    rpb = GmShape<MF, 2>::RPB;
    kst = MF::KST;
    per_cu = GmShape<MF, 2>::PER_CU;
}
static void dense_shape(int dtype, int &rpb, int &kst, int &per_cu) {
    switch (dtype) {
    case CW_IQ2_XXS: return shape_of<MIQ2_XXS>(rpb, kst, per_cu);
    case CW_IQ2_S: return shape_of<MIQ2_S>(rpb, kst, per_cu);
    case CW_IQ3_S: return shape_of<MIQ3_S>(rpb, kst, per_cu);
    case CW_MXFP4: return shape_of<MMXFP4>(rpb, kst, per_cu);
    case CW_Q8_0: return shape_of<MQ8_0>(rpb, kst, per_cu);
    case CW_Q2_K: return shape_of<MQ2_K>(rpb, kst, per_cu);
    case CW_IQ3_XXS: return shape_of<MIQ3_XXS>(rpb, kst, per_cu);
    case CW_IQ4_XS: return shape_of<MIQ4_XS>(rpb, kst, per_cu);
    default: return shape_of<MQ4_K>(rpb, kst, per_cu);
    }
}
// The split count S minimises the stages on the critical path: the launch's blocks (work items,
// padded as launch() pads them, times S) run in rounds of the resident blocks, and each block runs
// its items' ceil(n_st / S) stages one after another. (Filling the resident blocks exactly, as a
// first version did, left config 2's M = 512 at 768 blocks over 512 slots: 2 rounds of 6 stages
// where 1 round of 8 does.) Each 8 splits add a stage to the cost: the last split of a work item
// reads the partial rows 8 splits at a time (config 2 at M = 16: 16 splits of one stage measured
// 19.4 us, 8 splits of two 17.8). Ties go to fewer splits (less partial traffic).
int dense_splits(int rpb, int kst, int per_cu, int64_t m, int64_t n, int64_t k, int &split_st) {
    const int64_t tiles = (m + MF_MT - 1) / MF_MT;
    const int64_t items = gemm_items(tiles, rpb, n), res = resident_blocks(per_cu);
    const int64_t grid_x = items < res ? (items + 7) / 8 * 8 : res, per_block = (items + grid_x - 1) / grid_x;
    const int n_st = (int)((k / 32 + kst - 1) / kst);
    int best_s = 1;
    int64_t best = -1;
    for (int S = 1; S <= n_st; S++) {
        const int sst = (n_st + S - 1) / S;
        if ((n_st + sst - 1) / sst != S) continue;  // the same split as a smaller S
        if (S > 1 && (int64_t)S * m * n * 4 >= ((int64_t)1 << 31)) break;  // the partial rows stay under 2 GiB (32-bit offsets)
        const int64_t cost = (grid_x * S + res - 1) / res * per_block * sst + (S > 1 ? (S + 7) / 8 : 0);
        if (best < 0 || cost < best) {
            best = cost;
            best_s = S;
        }
    }
    split_st = (n_st + best_s - 1) / best_s;
    return best_s;
}
static int dense_splits(int dtype, int64_t m, int64_t n, int64_t k, int &split_st) {
    int rpb, kst, per_cu;
    dense_shape(dtype, rpb, kst, per_cu);
    return dense_splits(rpb, kst, per_cu, m, n, k, split_st);
}

// work items of the dense GEMM's launch
static int64_t dense_items(int dtype, int64_t m, int64_t n) {
    int rpb, kst, per_cu;
    dense_shape(dtype, rpb, kst, per_cu);
    return gemm_items((m + MF_MT - 1) / MF_MT, rpb, n);
}

size_t mfma_dense_workspace(int dtype, int64_t m, int64_t n, int64_t k) {
    int split_st;
    const int S = dense_splits(dtype, m, n, k, split_st);
    return al256(m * k * 2) + al256(m * 4) + al256((m + MF_MT - 1) / MF_MT * sizeof(MfTile)) + al256(4) +
           (S > 1 ? al256((size_t)S * m * n * 4) + al256((size_t)dense_items(dtype, m, n) * 4) : 0);
}

// Dense Q4_K QMatMul for 2..16 rows of x, one launch: block b takes weight rows
// 16b .. 16b+15 over the whole of k, its W waves a share of at most 2 super-blocks each (4 each
// measured 13.3 against 12.9 us for config 2 at M = 16: half the waves in flight), with all
// of a wave's loads (the rows' super-block headers and code bytes, and its activation fragments)
// issued at once: the persistent GEMM's per-stage window round trips and split-K partial rows
// cost ~12 us here for ~0.3 us of MFMA work. MFMA operands as in k_gmm: A = a token's 8 fp16
// activations (lane = token l16, K-group grp), B = a row's 8 codes sc*q (lane = row l16, K-group
// grp), and the minimum term as a second accumulator with codes -m; each super-block's sums are
// folded in f32 with the lane's row's d and dmin (a lane's 4 outputs share its row), the waves'
// partial tiles summed in LDS in wave order.
// X = uint16_t: rows packed by k_pack_f16 with one scale each (xs). X = float: the wave takes its share
// of x as it is, f32, and gives each token's 256 values of a super-block the power of two that keeps
// their largest in [2^14, 2^15) of fp16: one launch instead of two, for twice the bytes of x in every
// block (skinny_f32).
constexpr int SKINNY_SB = 2;  // super-blocks per wave
template <int W, typename X>
__global__ __launch_bounds__(64 * W) void k_skinny_q4k(const uint8_t *w, int64_t row_bytes, int n, int k, const X *x,
                                                       const float *xs, int m, float *y) {
    constexpr bool F32 = std::is_same_v<X, float>;
    // a wave's 16 rows x SKINNY_SB super-blocks, copied as 16-byte chunks (row r's bytes at r * RB)
    constexpr int RB = SKINNY_SB * 144, NCH = 16 * RB / 16, NI = (NCH + 63) / 64;
    __shared__ __align__(16) uint8_t wl[W][NI * 1024];
    __shared__ float part[W][16 * 16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, grp = lane >> 4;
    const int nsb = k / 256, s0 = wave * nsb / W, s1 = (wave + 1) * nsb / W;  // this wave's super-blocks
    const X *xr = x + (int64_t)min(l16, m - 1) * k + 8 * grp;
    // every load at once, from clamped rows and super-blocks (those past s1 are not used): the
    // weight bytes as whole 16-byte chunks of each row's run of super-blocks straight into LDS
    // (per-lane 8-byte pieces of 16 rows measured slower), then the activation fragments
#pragma unroll
    for (int t = 0; t < NI; t++) {
        const int c = min(64 * t + lane, NCH - 1), r = c / (RB / 16), piece = c - r * (RB / 16), j = piece / 9;
        dma16(w + (int64_t)min(blockIdx.x * 16 + r, n - 1) * row_bytes + 144 * min(s0 + j, nsb - 1) + 16 * (piece - 9 * j),
              lds_addr(&wl[wave][1024 * t]));
    }
    uint4 head[SKINNY_SB];
    uint2 qs[SKINNY_SB][4];
    constexpr int XL = F32 ? 16 : 8;  // 16-byte loads of x per super-block
    uint4 xl[SKINNY_SB][XL], xf[SKINNY_SB][8];
#pragma unroll
    for (int j = 0; j < SKINNY_SB; j++) {
        const int sb = min(s0 + j, nsb - 1);
#pragma unroll
        for (int c = 0; c < XL; c++) xl[j][c] = *(const uint4 *)(xr + 256 * sb + (F32 ? 32 * (c >> 1) + 4 * (c & 1) : 32 * c));
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XL * SKINNY_SB) : "memory");  // the chunks have landed
#pragma unroll
    for (int j = 0; j < SKINNY_SB; j++) {
        const uint8_t *blk = &wl[wave][l16 * RB + 144 * j];
        head[j] = *(const uint4 *)blk;  // d, dmin, the 12 scale bytes
#pragma unroll
        for (int c = 0; c < 4; c++) qs[j][c] = *(const uint2 *)(blk + 16 + 32 * c + 8 * grp);
    }
    // nothing moves across this point: the scheduler would otherwise sink later super-blocks'
    // loads behind earlier MFMAs (to save registers), one memory round trip per super-block
    __builtin_amdgcn_sched_barrier(0);
    f32x4 fin = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < SKINNY_SB; j++) {
        float inv[4] = {1.f, 1.f, 1.f, 1.f};  // 1 / scale of tokens 4*grp + i
        if constexpr (F32) {
            float mx = 0.f;
#pragma unroll
            for (int c = 0; c < XL; c++) {
                const float4 f = __builtin_bit_cast(float4, xl[j][c]);
                mx = fmaxf(mx, fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fmaxf(fabsf(f.z), fabsf(f.w))));
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16));  // over the token's four K-groups
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            int ex = 0;
            if (mx > 0.f && mx < INFINITY) {
                frexpf(mx, &ex);
                ex = min(15 - ex, 126);  // the scale stays finite and its inverse normal
            }
            const float sc = ldexpf(1.0f, ex), is = ldexpf(1.0f, -ex);
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const float4 f = __builtin_bit_cast(float4, xl[j][2 * kk]), g = __builtin_bit_cast(float4, xl[j][2 * kk + 1]);
                const f16x8 h = {(_Float16)(f.x * sc), (_Float16)(f.y * sc), (_Float16)(f.z * sc), (_Float16)(f.w * sc),
                                 (_Float16)(g.x * sc), (_Float16)(g.y * sc), (_Float16)(g.z * sc), (_Float16)(g.w * sc)};
                xf[j][kk] = __builtin_bit_cast(uint4, h);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) inv[i] = __shfl(is, 4 * grp + i);
        } else {
#pragma unroll
            for (int kk = 0; kk < 8; kk++) xf[j][kk] = xl[j][kk];
        }
        // no branch on the wave's super-block count: a branch here kept the compiler from issuing
        // the later super-blocks' loads before the first one's MFMAs
        f32x4 acc = {0.f, 0.f, 0.f, 0.f}, accm = {0.f, 0.f, 0.f, 0.f};
        const uint32_t sb12[3] = {head[j].y, head[j].z, head[j].w};
        auto sbyte = [&](int i) { return (sb12[i >> 2] >> (8 * (i & 3))) & 0xFFu; };
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            uint32_t sc, mn;  // the 6-bit scale and min of sub-block kk (get_scale_min_k4)
            if (kk < 4) {
                sc = sbyte(kk) & 63;
                mn = sbyte(kk + 4) & 63;
            } else {
                sc = (sbyte(kk + 4) & 0xF) | ((sbyte(kk - 4) >> 6) << 4);
                mn = (sbyte(kk + 4) >> 4) | ((sbyte(kk) >> 6) << 4);
            }
            const int sh = 4 * (kk & 1);
            const uint2 q = qs[j][kk >> 1];
            const uint4 codes = fma4(bytes_plus_1024((q.x >> sh) & 0x0F0F0F0Fu, (q.y >> sh) & 0x0F0F0F0Fu), splat_f16f((float)sc),
                                     splat_f16f(-1024.0f * (float)sc));
            const uint32_t mv = splat_f16f(-(float)mn);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(xf[j][kk]), as_f16x8(codes), acc, 0, 0, 0);
            accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(xf[j][kk]), as_f16x8(make_uint4(mv, mv, mv, mv)), accm, 0, 0, 0);
        }
        const bool live = s0 + j < s1;
        const float d = live ? h2f(head[j].x & 0xFFFF) : 0.f, dmin = live ? h2f(head[j].x >> 16) : 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) fin[i] += inv[i] * (d * acc[i] + dmin * accm[i]);
    }
    // lane: tokens 4*grp + i of weight row l16
#pragma unroll
    for (int i = 0; i < 4; i++) part[wave][(4 * grp + i) * 16 + l16] = fin[i];
    __syncthreads();
    for (int e = threadIdx.x; e < 256; e += 64 * W) {
        const int t = e >> 4, r = blockIdx.x * 16 + (e & 15);
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < W; q++) v += part[q][e];
        if (t < m && r < n) y[(int64_t)t * n + r] = F32 ? v : v * xs[t];
    }
}

// Where the GEMM takes x as f32 rather than packed by a launch before it (4 blocks, 4 us): one block per
// CU at most, and at most 128 KB of x per block. us per call, packed / f32: 4096 x 4096 at 2 rows 9.2 / 7.8,
// at 8 rows 10.3 / 9.2, 4096 x 2048 at 16 rows 8.5 / 7.5, 4096 x 1024 at 16 rows 7.3 / 5.7, 512 x 512 at 16
// rows 6.6 / 4.8. Past it the loads of x cost as much as the launch or more: 4096 x 4096 at 16 rows 12.1 /
// 11.8 (equal within the runs' spread), 4096 x 3072 at 16 rows 10.8 / 11.5, 8192 x 4096 at 2 rows 12.6 / 14.3, at 16 rows 16.3 / 21.4,
// 5120 x 2048 at 16 rows 10.5 / 11.4. (A 16-wave block, k above 4,096, would not have the registers.)
static bool skinny_f32(int n, int waves, int m) { return n <= 16 * resident_blocks(1) && m * waves * SKINNY_SB * 256 <= 32768; }

// 2..16 rows of Q4_K x: k_skinny_q4k, after the pack (fp16 activations and their scales) if it takes packed rows
static int dense_skinny_q4k(const uint8_t *w, int64_t row_bytes, int n, int k, const float *x, int m, float *y, uint16_t *x16,
                            float *xs, hipStream_t s) {
    const int nsb = k / 256, need = (nsb + SKINNY_SB - 1) / SKINNY_SB;
    const int waves = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : need <= 8 ? 8 : 16;
    if (need > 16) return set_error(CW_ENOTSUP, "qmatmul: k %d above %d for the skinny Q4_K path", k, 16 * SKINNY_SB * 256);
    const dim3 grid((unsigned)((n + 15) / 16)), block(64 * waves);
    if (waves <= 8 && skinny_f32(n, waves, m)) {
#define CW_SKINNY(W) hipLaunchKernelGGL((k_skinny_q4k<W, float>), grid, block, 0, s, w, row_bytes, n, k, x, nullptr, m, y)
        if (waves == 1) CW_SKINNY(1);
        else if (waves == 2) CW_SKINNY(2);
        else if (waves == 4) CW_SKINNY(4);
        else CW_SKINNY(8);
#undef CW_SKINNY
        return check_launch("k_skinny_q4k");
    }
    int rc;
    if ((rc = pack_rows_f16(x, m, k, k, x16, xs, s, nullptr, K_NATURAL))) return rc;
#define CW_SKINNY(W) hipLaunchKernelGGL((k_skinny_q4k<W, uint16_t>), grid, block, 0, s, w, row_bytes, n, k, x16, xs, m, y)
    if (waves == 1) CW_SKINNY(1);
    else if (waves == 2) CW_SKINNY(2);
    else if (waves == 4) CW_SKINNY(4);
    else if (waves == 8) CW_SKINNY(8);
    else CW_SKINNY(16);
#undef CW_SKINNY
    return check_launch("k_skinny_q4k");
}

int mfma_dense(int dtype, const uint8_t *w, int64_t row_bytes, int n, int k, const float *x, int m, float *y, void *ws,
               size_t ws_bytes, hipStream_t s) {
    const size_t need = mfma_dense_workspace(dtype, m, n, k);
    if (ws_bytes < need || !ws) return set_error(CW_EINVAL, "qmatmul: workspace of %zu bytes, %zu needed", ws_bytes, need);
    int split_st;
    const int S = dense_splits(dtype, m, n, k, split_st);
    uint8_t *p = (uint8_t *)ws;
    uint16_t *x16 = (uint16_t *)p; p += al256((size_t)m * k * 2);
    float *xs = (float *)p; p += al256((size_t)m * 4);
    // (its rows are copied as 16-byte chunks: a matrix off 16-byte alignment takes the GEMM below)
    if (dtype == CW_Q4_K && m <= 16 && ((uintptr_t)w & 15) == 0) return dense_skinny_q4k(w, row_bytes, n, k, x, m, y, x16, xs, s);
    MfTile *tiles = (MfTile *)p; p += al256((size_t)(m + MF_MT - 1) / MF_MT * sizeof(MfTile));
    int *n_tiles = (int *)p; p += al256(4);
    float *part = nullptr;
    int *cnt = nullptr;
    if (S > 1) {
        part = (float *)p;
        p += al256((size_t)S * m * n * 4);
        cnt = (int *)p;
    }
    // one launch packs x, writes the tile list and zeroes the split counters
    const PackExtra extra = {tiles, n_tiles, m, cnt, S > 1 ? (int)dense_items(dtype, m, n) : 0};
    int rc;
    if ((rc = pack_rows_f16(x, m, k, k, x16, xs, s, &extra, k_order(dtype)))) return rc;
    MfArgs a = {};
    a.w0 = w;
    a.s0 = 0;
    a.row_bytes = row_bytes;
    a.n = n;
    a.k = k;
    a.a16 = x16;
    a.ascale = xs;
    a.lda = k;
    a.tiles = tiles;
    a.n_tiles = n_tiles;
    a.K = 1;
    a.dn = S > 1 ? part : y;
    a.split_st = S > 1 ? split_st : 0;
    a.split_stride = (int64_t)m * n;
    a.split_cnt = cnt;
    a.y = y;
    return by_fmt<2>(dtype, a, (m + MF_MT - 1) / MF_MT, S, s);
}

int mfma_gateup(int dtype, const MfArgs &a, int tiles_max, hipStream_t s) { return by_fmt<0>(dtype, a, tiles_max, 1, s); }
int mfma_down(int dtype, const MfArgs &a, int tiles_max, hipStream_t s) { return by_fmt<1>(dtype, a, tiles_max, 1, s); }

}  // namespace cw
