// Attention of one query row over one head by two waves, shared by the batch-1 step kernels
// (per-layer launches and the resident step), so that both sum in the same order.
#pragma once
#include "device.hpp"
#include "kernels.hpp"

namespace mlg {

// Wave q of the pair (batch 1, head groups of <= 2 heads) takes the SPL-key groups 2 i + q: pass u of its chunk c covers keys
// SPL (2 (c U2 + u) + q) + split.  Each wave keeps an online softmax over its keys and
// leaves its partial in LDS: po[HD] = sum_j p_j v_j (unnormalized), pml = (max, sum_j p_j)
// with p_j = exp(s_j - max).  attn_combine2 then rescales the two partials to their common
// max and divides: the same keys and the same order of sums whichever kernel runs it.
constexpr int kHalfU = 4;                  // passes per chunk of a half
constexpr int kHalfSlot = 128 + 2;         // floats of one wave's partial (HD <= 128)
__host__ __device__ constexpr int half_key(int spl, int c, int u, int q) { return spl * (2 * (c * kHalfU + u) + q); }

template <int HD, class LoadF>
__device__ __forceinline__ void attn_half(int n, int q, const float4 &qa, const float4 &qb, const uint4 (&kr)[kHalfU],
                                          const uint4 (&vr)[kHalfU], LoadF &&load, float *wsc, float *slot) {
    constexpr int TPK = HD / 8, SPL = 64 / TPK;
    const int lane = threadIdx.x & 63, sub = lane % TPK, split = lane / TPK;
    float m = -INFINITY, l = 0.f;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c = 0; half_key(SPL, c, 0, q) < n; ++c) {  // wave-uniform; chunk 0 is in flight
        if (c) load(c);
        float sc[kHalfU];
        float cmax = -INFINITY;
#pragma unroll
        for (int u = 0; u < kHalfU; ++u) {
            float s = h2f(kr[u].x) * qa.x;
            s = fmaf(h2f(kr[u].x >> 16), qa.y, s);
            s = fmaf(h2f(kr[u].y), qa.z, s);
            s = fmaf(h2f(kr[u].y >> 16), qa.w, s);
            s = fmaf(h2f(kr[u].z), qb.x, s);
            s = fmaf(h2f(kr[u].z >> 16), qb.y, s);
            s = fmaf(h2f(kr[u].w), qb.z, s);
            s = fmaf(h2f(kr[u].w >> 16), qb.w, s);
            s = group_sum<TPK>(s);
            sc[u] = half_key(SPL, c, u, q) + split < n ? s : -INFINITY;
            cmax = fmaxf(cmax, sc[u]);
        }
        const float mnew = fmaxf(m, wave_max(cmax));  // finite: the chunk's first key is valid
        const float r = expf(m - mnew);
        l *= r;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] *= r;
#pragma unroll
        for (int u = 0; u < kHalfU; ++u) {
            const bool in = half_key(SPL, c, u, q) + split < n;
            const float pj = in ? expf(sc[u] - mnew) : 0.f;
            l += pj;
            const uint32_t wv[4] = {in ? vr[u].x : 0u, in ? vr[u].y : 0u, in ? vr[u].z : 0u, in ? vr[u].w : 0u};
#pragma unroll
            for (int q2 = 0; q2 < 4; ++q2) {
                acc[2 * q2] = fmaf(pj, h2f(wv[q2]), acc[2 * q2]);
                acc[2 * q2 + 1] = fmaf(pj, h2f(wv[q2] >> 16), acc[2 * q2 + 1]);
            }
        }
        m = mnew;
    }
    // every lane of a split holds that split's sum; count each split once
    const float lsum = wave_sum(sub == 0 ? l : 0.f);
#pragma unroll
    for (int e = 0; e < 8; ++e) wsc[lane * 8 + e] = acc[e];
    __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's LDS writes are done
    __builtin_amdgcn_wave_barrier();
    for (int e = lane; e < HD; e += 64) {
        float o = 0.f;
#pragma unroll
        for (int s2 = 0; s2 < SPL; ++s2) o += wsc[(s2 * TPK + e / 8) * 8 + e % 8];
        slot[e] = o;
    }
    if (lane == 0) {
        slot[HD] = m;  // -inf when this wave had no key
        slot[HD + 1] = lsum;
    }
}

// out[e] of the pair from the partials of its two waves (after a workgroup barrier)
template <int HD>
__device__ __forceinline__ void attn_combine2(const float *s0, const float *s1, float *out) {
    const int lane = threadIdx.x & 63;
    const float m0 = s0[HD], m1 = s1[HD], M = fmaxf(m0, m1);  // m0 finite: wave 0 has key 0
    const float e0 = expf(m0 - M), e1 = expf(m1 - M);
    const float inv = 1.f / (e0 * s0[HD + 1] + e1 * s1[HD + 1]);
    for (int e = lane; e < HD; e += 64) out[e] = (e0 * s0[e] + e1 * s1[e]) * inv;
}

}  // namespace mlg
