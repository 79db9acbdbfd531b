// Router logits: logits[t][e] = x[t] . W[e] (+ bias[e]) for the router weight W (E x h), f32 or
// f16 weights, f32 activations and accumulation.
//
// Replaces the engine's gate Linear (crates/engine/src/experts.rs:2428, 2577; the weight is
// dequantized to f32 at load, model_next.rs:1036; gpt-oss adds a bias, model_gptoss.rs:168-175)
// and its f16 decode variant cw_mv_f16 (crates/engine/src/fuse_kernel.rs:160-178, 537-559).
//
//  - A few tokens (decode): one wave per expert row; lanes stride the row in 4-element pieces,
//    each piece of W read once and used for every token; a DPP wave sum per token.
//  - Many tokens (prefill): 32 x 32 tiles on the f32 matrix instruction, K in chunks through LDS.
#include <atomic>

#include "cw_common.h"
#include "cw_router.h"
#include "cw_wave.h"

namespace cw {

template <class WT>
__device__ __forceinline__ float4 load4(const WT *p);
template <>
__device__ __forceinline__ float4 load4<float>(const float *p) {
    return *(const float4 *)p;
}
template <>
__device__ __forceinline__ float4 load4<_Float16>(const _Float16 *p) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 v = *(const h4 *)p;
    return make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
}

constexpr int ROUTER_FEW = 8;  // tokens up to which the per-row kernel runs

template <class WT, int TT>
__global__ __launch_bounds__(256) void k_router_rows(const WT *w, const float *bias, const float *x, int E, int h, int T,
                                                     float *logits) {
    const int lane = threadIdx.x & 63, e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= E) return;  // whole wave
    const WT *wr = w + (int64_t)e * h;
    float acc[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) acc[t] = 0.f;
    for (int k = 4 * lane; k < h; k += 256) {
        const float4 a = load4<WT>(wr + k);
#pragma unroll
        for (int t = 0; t < TT; t++) {
            if (t >= T) break;
            const float4 b = *(const float4 *)(x + (int64_t)t * h + k);
            acc[t] = fmaf(a.x, b.x, fmaf(a.y, b.y, fmaf(a.z, b.z, fmaf(a.w, b.w, acc[t]))));
        }
    }
    const float be = bias ? bias[e] : 0.f;
#pragma unroll
    for (int t = 0; t < TT; t++) {
        if (t >= T) break;
        const float s = wave_sum(acc[t]);
        if (lane == 0) logits[(int64_t)t * E + e] = s + be;
    }
}

// 32 tokens x 32 experts per block, one 16 x 16 tile per wave on v_mfma_f32_16x16x4_f32, whose sum
// is the chain fma(a_k, b_k, acc) over ascending k, one rounding each (subnormals kept): the logits
// are those of a scalar loop over k, bit for bit, and do not depend on the tile. K goes through LDS in
// chunks of 256, the next chunk's loads in flight during this one's 64 MFMAs; rows 260 floats apart
// put the 64 lanes of a fragment read on distinct banks. What bounds it is that chain (32 cycles per
// 4 weights, 6.8 us for 2,048); 64 x 64 tiles on the VALU (10 blocks for 301 tokens x 128 experts, a
// round trip to memory per 32 of K) took 122 us where this takes 19.6 (1,500 x 256: 147 and 41.6).
constexpr int RT = 32, RKC = 256, RLD = RKC + 4;
template <class WT>
__global__ __launch_bounds__(256) void k_router_tiles(const WT *w, const float *bias, const float *x, int E, int h, int T,
                                                      float *logits) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) float rs[];  // two buffers of RT token rows, then RT expert rows
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, grp = lane >> 4;
    const int e0 = blockIdx.x * RT, t0 = blockIdx.y * RT;
    // wave w copies rows w, w + 4, ... of the chunk, lane l 4 floats from 4 l (rows and columns past
    // the matrices: a clamped address, zeros stored)
    float4 v[2 * RT / 4];
    auto fetch = [&](int kc) __attribute__((always_inline)) {
        const int k = kc + 4 * lane, kk = k < h ? k : h - 4;
#pragma unroll
        for (int i = 0; i < 2 * RT / 4; i++) {
            const int r = 4 * i + wave;
            if (r < RT) v[i] = *(const float4 *)(x + (int64_t)min(t0 + r, T - 1) * h + kk);
            else v[i] = load4<WT>(w + (int64_t)min(e0 + r - RT, E - 1) * h + kk);
        }
        if (k >= h) {
#pragma unroll
            for (int i = 0; i < 2 * RT / 4; i++) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    fetch(0);
    const int tr = 16 * (wave & 1), er = 16 * (wave >> 1);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int kc = 0, b = 0; kc < h; kc += RKC, b ^= 1) {
        float *buf = rs + b * 2 * RT * RLD;
#pragma unroll
        for (int i = 0; i < 2 * RT / 4; i++) *(float4 *)(buf + (4 * i + wave) * RLD + 4 * lane) = v[i];
        __syncthreads();  // (the other buffer is refilled only after the next one)
        if (kc + RKC < h) fetch(kc + RKC);
        const float *xa = buf + (tr + l16) * RLD + grp, *wb = buf + (RT + er + l16) * RLD + grp;
#pragma unroll
        for (int j = 0; j < RKC / 4; j++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[4 * j], wb[4 * j], acc, 0, 0, 0);
    }
    const int e = e0 + er + l16;
    if (e >= E) return;
    const float be = bias ? bias[e] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int t = t0 + tr + 4 * grp + i;
        if (t < T) logits[(int64_t)t * E + e] = acc[i] + be;
    }
}

template <class WT>
static int launch(const void *w, const float *bias, const float *x, int E, int h, int T, float *logits, hipStream_t s) {
    const WT *wt = (const WT *)w;
    if (T <= ROUTER_FEW) {
        const dim3 grid((E + 3) / 4);
#define CW_ROWS(N) \
    if (T <= N) { hipLaunchKernelGGL((k_router_rows<WT, N>), grid, dim3(256), 0, s, wt, bias, x, E, h, T, logits); return check_launch("k_router_rows"); }
        CW_ROWS(1) CW_ROWS(2) CW_ROWS(4) CW_ROWS(8)
#undef CW_ROWS
    }
    // dynamic LDS above 64 KB, opted into once per device
    constexpr int MAX_DEVICES = 64;
    constexpr size_t lds = 2 * 2 * RT * RLD * sizeof(float);
    static std::atomic<bool> lds_set[MAX_DEVICES];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) dev = 0;
    if (!lds_set[dev].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute((const void *)k_router_tiles<WT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return set_error(CW_EHIP, "router: cannot reserve %zu bytes of LDS", lds);
        lds_set[dev].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((k_router_tiles<WT>), dim3((E + RT - 1) / RT, (T + RT - 1) / RT), dim3(256), lds, s, wt, bias, x, E, h, T, logits);
    return check_launch("k_router_tiles");
}

int router_logits(int wdtype, const void *w, int E, int h, const float *bias, const float *x, int T, float *logits,
                  hipStream_t s) {
    if (T == 0 || E == 0) return CW_OK;
    if (h % 4) return set_error(CW_ENOTSUP, "router: hidden %d is not a multiple of 4", h);
    switch (wdtype) {
    case CW_F32: return launch<float>(w, bias, x, E, h, T, logits, s);
    case CW_F16: return launch<_Float16>(w, bias, x, E, h, T, logits, s);
    default: return set_error(CW_ENOTSUP, "router: weight dtype %d (f32 or f16 only)", wdtype);
    }
}

}  // namespace cw
