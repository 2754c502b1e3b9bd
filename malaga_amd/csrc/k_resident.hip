// All decoder layers of a batch-1 step in one resident launch (src/model.rs:552-612 for
// one row; the static step of src/graph.rs).
//
// What bounds the step at batch 1 is not the weights (112 MB of layers, 14 us at 8 TB/s) but
// the chain of dependent launches: five per layer, each a dispatch and the read of what the
// previous one wrote (28.5 us per layer).  Here the workgroups stay resident for the whole
// step and hand vectors on through memory, and every weight a workgroup will multiply is in
// its registers before the vector it multiplies arrives.
//
// Hand-over.  A value travels as one 8-byte word { f32 value, launch tag } written and read
// with relaxed agent-scope atomics: the tag says that the value is this launch's, so no
// fence, counter or barrier between workgroups is needed, and every vector of every layer
// has words of its own, so nothing is overwritten within a launch.  1024 words from 128
// workgroups to 128 workgroups take 1.5 us including the workgroup's own reduction (256
// workgroups: 2.0 us, so 128 share the rows).  A layer of the 600M model takes 17.5 us this
// way (q4_K, 21 keys): seven hand-overs of 0.9 .. 1.5 us, three LayerNorms of 0.5, products
// 4.5 and the two attentions 2.4 us; a sentence of 21 ids in and 18 tokens out 7.85 -> 5.47 ms.
//
// Roles.  Workgroups 0 .. H-1 own one attention head each: its self attention and, with the
// head's 64 rows of the cross q projection, its cross attention.  The other kResPlain own
// 1 / kResPlain of the rows of every other projection.  In both, waves 8..11 gather vectors,
// keep the residual stream (a copy in each workgroup, the same operations in the same order)
// and normalize; waves 0..7 hold weights and keys and multiply.  A wave's loads complete in
// order, so a wave that did both would wait for its weights at every poll (29 us per layer).
// A job's weights for the next layer are requested as soon as this layer's have been used,
// so they have most of a layer's time to arrive.
//
// Every wait is bounded: a wave that runs out of polls (the workgroups are not all resident,
// for instance behind other long kernels) raises *flag and goes on without waiting, so the
// launch always ends; the caller sees the flag and decodes again with the other kernels.
#include "dequant.hpp"
#include "gemv_core.hpp"
#include "kernels.hpp"

namespace mlg {

namespace {

constexpr int kResWaves = 8;     // waves 0..7 multiply and attend, waves 8..11 gather
constexpr int kResGather = 256;  // gathering threads (12 waves of 168 registers: with 16 of 128 the
                                 // multiplying waves spill)
constexpr int kResGatherWaves = kResGather / 64;
constexpr int kResThreads = 64 * kResWaves + kResGather;
constexpr int kResPlain = 128;  // workgroups that share the projections' rows
constexpr int kResMaxD = 1024, kResMaxF = 4096, kResHd = 64, kResMaxLayers = 32;

using word_t = unsigned long long;

__device__ __forceinline__ void put(word_t *p, float v, uint32_t tag) {
    __hip_atomic_store(p, (word_t(tag) << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct ResArgs {
    const ResLayer *layers;
    int L, d, f, H;
    word_t *words;        // [L][8 d + f]: q k v | att | out | cross att | cross out | ffn u | down
    uint32_t *epoch;      // tag of this launch; + 1 at its end
    uint32_t *flag;       // set when a wait ran out
    uint32_t spins;
    // input: E[ids[0]] * emb_scale + pos[*step + pos_base], or a copied source token
    const uint8_t *eq, *es, *ed;
    const uint32_t *ids;
    uint32_t elast;
    const float *src_emb;
    const uint32_t *src_row;
    const float *pos;
    uint32_t pos_base;
    float emb_scale, eps;
    const uint32_t *step, *lens;
    __half *kv;           // self caches: layer l's K at 2 l self_pair, V behind it, [H][m][hd]
    const __half *ckv;    // cross K/V likewise, [H][s][hd]
    size_t self_pair, cross_pair;
    int m, s;
    float *x_out, *y;     // the residual stream and the last FFN output, for the LM head
};

// words of layer l
struct Words {
    word_t *q, *att, *out, *catt, *cout, *u, *down;
};
__device__ __forceinline__ Words words_of(const ResArgs &a, int l) {
    word_t *p = a.words + size_t(l) * (8 * a.d + a.f);
    return {p, p + 3 * a.d, p + 4 * a.d, p + 5 * a.d, p + 6 * a.d, p + 8 * a.d, p + 7 * a.d};
}

// A wave's bounded wait for N words p[0], p[stride], ..: every lane's values, or whatever is
// there once the polls have run out (then dead: later waits look once)
struct Waiter {
    uint32_t tag, spins;
    uint32_t *flag;
    bool dead;
    template <int N>
    __device__ __forceinline__ void get(const word_t *p, int stride, float (&v)[N]) {
        word_t w[N];
        for (uint32_t i = 0;; ++i) {
#pragma unroll
            for (int k = 0; k < N; ++k) w[k] = __hip_atomic_load(p + k * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bool ok = true;
#pragma unroll
            for (int k = 0; k < N; ++k) ok &= uint32_t(w[k] >> 32) == tag;
            if (__all(ok)) break;
            if (dead || i >= spins) {
                if (!dead) *flag = 1u;
                dead = true;
                break;
            }
        }
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = __uint_as_float(uint32_t(w[k]));
    }
};

// Vectors in LDS are kept as the lanes that multiply them read them, 16 bytes per lane and
// instruction from 1 KB of whole rows of banks:
//   q4_K / q5_K rows: d / 16 lanes of 16 values, lane 16 kb + 4 g + qt the bytes 8 qt .. 8 qt + 7
//     of 64-value group g of block kb (low nibbles: x[256 kb + 64 g + 8 qt ..], high: + 32);
//   q6_K rows (FFN down): K / 64 lanes of 64 values, the chunks of load_chunk<q6_K>.
__device__ __forceinline__ int pos_k4(int k, int lanes) {
    const int lane = (k >> 6) * 4 + ((k >> 3) & 3), v = ((k >> 5) & 1) * 8 + (k & 7);
    return (v >> 2) * (4 * lanes) + 4 * lane + (v & 3);
}
__device__ __forceinline__ int pos_k6(int k, int lanes) {
    const int lane = (k >> 8) * 4 + ((k >> 7) & 1) * 2 + ((k >> 4) & 1), e = ((k >> 5) & 3) * 16 + (k & 15);
    return (e >> 2) * (4 * lanes) + 4 * lane + (e & 3);
}

// A pointer that is the same in every lane, as a scalar in the global address space: loads then
// take a 32-bit lane offset, and (the layer table being read from LDS) are not flat loads,
// which the barriers' LDS waits would wait for too.
typedef const __attribute__((address_space(1))) uint8_t *gptr;
__device__ __forceinline__ gptr uniform(const void *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v)), hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
    return reinterpret_cast<gptr>((uint64_t(hi) << 32) | lo);
}
__device__ __forceinline__ uint4 ld16(gptr p) {
    const u32x4_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t *>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 ld8(gptr p) {
    const u32x2_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x2_t *>(p);
    return make_uint2(v.x, v.y);
}
__device__ __forceinline__ float ldf(gptr p) { return *reinterpret_cast<const __attribute__((address_space(1))) float *>(p); }

// sum over aligned groups of W = 16, 32 or 64 lanes, in every lane
template <int W>
__device__ __forceinline__ float lanes_sum(float v) {
    v += dpp_mov<kDppXor1>(v);
    v += dpp_mov<kDppXor2>(v);
    v += dpp_mov<kDppHalfMirror>(v);
    v += dpp_mov<kDppMirror>(v);
    if constexpr (W >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    if constexpr (W >= 64) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    return v;
}

struct XK4 {  // a lane's 16 values and the sums of its two halves
    float x[16], s[2];
    __device__ __forceinline__ void load(const float *xs, int lanes, int lane) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = *reinterpret_cast<const float4 *>(xs + 4 * lanes * i + 4 * lane);
            x[4 * i] = v.x, x[4 * i + 1] = v.y, x[4 * i + 2] = v.z, x[4 * i + 3] = v.w;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float *p = x + 8 * h;
            s[h] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        }
    }
};

// NP passes of 8 RPW rows (D / 16 = 2^LG lanes per row, RPW rows per wave) from row0 on, `rows`
// in all.  A wave past the last row takes the last RPW rows (or all there are) again.
template <int T, int NP, int D>
struct RowsK4 {
    static constexpr int LG = D == 1024 ? 6 : D == 512 ? 5 : 4, RPW = 64 >> LG, K = D;
    static constexpr int B = T == GGML_Q4_K ? 144 : 176;
    uint4 h[NP];
    uint2 q[NP], qh[NP];  // qh: q5_K's fifth bits
    __device__ __forceinline__ static int first_row(int p, int rows, int wave) {
        return min((p * kResWaves + wave) * RPW, max(rows - RPW, 0));
    }
    __device__ __forceinline__ void load(const ResMat &mt, int row0, int rows, int wave, int lane) {
        __builtin_amdgcn_sched_barrier(0);  // the registers' last values have been used
        const int cl = lane & ((1 << LG) - 1), g = (cl >> 2) & 3, qt = cl & 3, rb = (K >> 8) * B;
        const uint32_t off = uint32_t(min(lane >> LG, rows - 1) * rb + (cl >> 4) * B), oq = off + (B - 128) + 32 * g + 8 * qt;
        const gptr m0 = uniform(mt.q) + size_t(row0) * rb;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const gptr base = m0 + first_row(p, rows, wave) * rb;
            h[p] = ld16(base + off);
            q[p] = ld8(base + oq);
            if constexpr (T == GGML_Q5_K) qh[p] = ld8(base + off + 16 + 8 * qt);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // h becomes (d sc0, d sc1, dmin m0, dmin m1) of the lane's two sub-blocks (q4_K: d sc1 / 16,
    // whose quants run() leaves 16 times as large).  Done while the wave has nothing to wait
    // for but its vector, so that the scales cost nothing once that is there.
    __device__ __forceinline__ void prepare(int lane) {
        const int g = ((lane & ((1 << LG) - 1)) >> 2) & 3, sh0 = 8 * ((2 * g) & 3), sh1 = sh0 + 8;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const uint4 hd = h[p];
            const float d = h2f(hd.x), dmin = h2f(hd.x >> 16);
            auto decode = [&](int sh, float &sc, float &mn) {
                const uint32_t B0 = hd.y >> sh, B1 = hd.z >> sh, B2 = hd.w >> sh;
                sc = d * float(g >= 2 ? ((B2 & 15u) | ((B0 >> 2) & 48u)) : (B0 & 63u));
                mn = dmin * float(g >= 2 ? (((B2 >> 4) & 15u) | ((B1 >> 2) & 48u)) : (B1 & 63u));
            };
            float sc0, m0, sc1, m1;
            decode(sh0, sc0, m0);
            decode(sh1, sc1, m1);
            if constexpr (T == GGML_Q4_K) sc1 *= 0.0625f;
            h[p] = make_uint4(__float_as_uint(sc0), __float_as_uint(sc1), __float_as_uint(m0), __float_as_uint(m1));
        }
        // here, not where the values are used (behind the barrier)
#pragma unroll
        for (int p = 0; p < NP; ++p) asm volatile("" : "+v"(h[p].x), "+v"(h[p].y), "+v"(h[p].z), "+v"(h[p].w));
    }
    // store(row of the job, sum) by the first lane of each row
    template <class F>
    __device__ __forceinline__ void run(const float *xs, int rows, int wave, int lane, F &&store) const {
        const int cl = lane & ((1 << LG) - 1), g = (cl >> 2) & 3;
        XK4 X;
        X.load(xs, 1 << LG, cl);
        float v[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            uint2 qp = q[p];
            // pass p starts when pass p - 2 has its sum: all of them expanded at once exceed
            // the registers
            if (p >= 2) asm volatile("" : "+v"(qp.x), "+v"(qp.y), "+v"(v[p - 2]));
            float al[2], ah[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const uint32_t w = u ? qp.y : qp.x;
                uint32_t lo = w & 0x0F0F0F0Fu, hi = w & 0xF0F0F0F0u;  // hi: 16 * nibble
                if constexpr (T == GGML_Q5_K) {
                    const uint32_t hb = u ? qh[p].y : qh[p].x;
                    lo |= ((hb >> (2 * g)) & 0x01010101u) << 4;
                    hi = ((w >> 4) & 0x0F0F0F0Fu) | (((hb >> (2 * g + 1)) & 0x01010101u) << 4);
                }
                al[u] = dot4u8(lo, X.x + 4 * u, 0.f);
                ah[u] = dot4u8(hi, X.x + 8 + 4 * u, 0.f);
            }
            const float m = fmaf(__uint_as_float(h[p].z), X.s[0], __uint_as_float(h[p].w) * X.s[1]);
            v[p] = fmaf(__uint_as_float(h[p].x), al[0] + al[1], __uint_as_float(h[p].y) * (ah[0] + ah[1])) - m;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            v[p] = lanes_sum<(1 << LG)>(v[p]);
            if ((p * kResWaves + wave) * RPW < rows && cl == 0 && (lane >> LG) < rows)
                store(first_row(p, rows, wave) + (lane >> LG), v[p]);
        }
    }
};

// one q6_K row per wave, row0 + wave
struct RowK6 {
    Raw<GGML_Q6_K> w;
    __device__ __forceinline__ void load(const ResMat &mt, int K, int row0, int rows, int wave, int lane) {
        __builtin_amdgcn_sched_barrier(0);
        const int c = min(lane, K / 64 - 1), h2 = (c >> 1) & 1, i = c & 1;  // as load_chunk<q6_K>
        const size_t blk = size_t(row0 + min(wave, rows - 1)) * (K / 256);
        const gptr qb = uniform(mt.q) + blk * 192 + uint32_t((c >> 2) * 192 + 64 * h2 + 16 * i);
        w.a = ld16(qb);
        w.b = ld16(qb + 32);
        w.h = ld16(uniform(mt.q) + blk * 192 + uint32_t((c >> 2) * 192 + 128 + 32 * h2 + 16 * i));
        const uint2 sc = ld8(uniform(mt.s) + blk * 16 + uint32_t((c >> 2) * 16 + 8 * h2));
        w.e0 = sc.x, w.e1 = sc.y;
        w.c.x = *reinterpret_cast<const __attribute__((address_space(1))) unsigned short *>(uniform(mt.d) + blk * 2 +
                                                                                         uint32_t((c >> 2) * 2));
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ float run(const float *xs, int K, int lane) const {
        const int lanes = K / 64, c = min(lane, lanes - 1), i = c & 1;
        const float sc[4] = {float(int8_t(w.e0 >> (8 * i))), float(int8_t(w.e0 >> (8 * i + 16))),
                             float(int8_t(w.e1 >> (8 * i))), float(int8_t(w.e1 >> (8 * i + 16)))};
        const uint32_t A[4] = {w.a.x, w.a.y, w.a.z, w.a.w}, B[4] = {w.b.x, w.b.y, w.b.z, w.b.w},
                       H[4] = {w.h.x, w.h.y, w.h.z, w.h.w};
        float q[4] = {0.f, 0.f, 0.f, 0.f}, sx[4] = {0.f, 0.f, 0.f, 0.f};
        int o = 4 * c;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (u == 2) asm volatile("" : "+v"(o), "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]));  // half of x at a time
            const uint32_t w4[4] = {(A[u] & 0x0F0F0F0Fu) | ((H[u] << 4) & 0x30303030u),
                                    (B[u] & 0x0F0F0F0Fu) | ((H[u] << 2) & 0x30303030u),
                                    ((A[u] >> 4) & 0x0F0F0F0Fu) | (H[u] & 0x30303030u),
                                    ((B[u] >> 4) & 0x0F0F0F0Fu) | ((H[u] >> 2) & 0x30303030u)};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float4 v = *reinterpret_cast<const float4 *>(xs + 4 * lanes * (4 * k + u) + o);
                const float x[4] = {v.x, v.y, v.z, v.w};
                q[k] = dot4u8(w4[k], x, q[k]);
                sx[k] += (v.x + v.y) + (v.z + v.w);
            }
        }
        float acc = h2f(w.c.x) * (sc[0] * (q[0] - 32.f * sx[0]) + sc[1] * (q[1] - 32.f * sx[1]) +
                                  sc[2] * (q[2] - 32.f * sx[2]) + sc[3] * (q[3] - 32.f * sx[3]));
        if (lane >= lanes) acc = 0.f;
        return lanes_sum<64>(acc);
    }
};

// K and V of one key, 8 dimensions per lane
struct KeyRegs {
    uint4 k, v;
};
// sum over the lanes that share lane % 8
__device__ __forceinline__ float sum_splits(float v) {
    v += dpp_mov<0x128>(v);  // row_ror:8
    const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
    const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

// Attention of one query over n keys by the 8 waves of a workgroup: wave w takes keys
// 64 c + 8 w + split, an online softmax per wave, its partial (64 sums, max, weight sum) to
// slot w.  key(j): K and V of key j (the first round's are passed in).
template <class KeyF>
__device__ __forceinline__ void attn_partial(int n, int wave, int lane, const float *q, KeyRegs kv, KeyF &&key,
                                             float *slot) {
    const int sub = lane & 7, split = lane >> 3;
    const float4 qa = *reinterpret_cast<const float4 *>(q + 8 * sub), qb = *reinterpret_cast<const float4 *>(q + 8 * sub + 4);
    float m = -INFINITY, l = 0.f;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j0 = 8 * wave; j0 < n; j0 += 8 * kResWaves) {  // wave-uniform
        if (j0 != 8 * wave) kv = key(min(j0 + split, n - 1));
        float s = h2f(kv.k.x) * qa.x;
        s = fmaf(h2f(kv.k.x >> 16), qa.y, s);
        s = fmaf(h2f(kv.k.y), qa.z, s);
        s = fmaf(h2f(kv.k.y >> 16), qa.w, s);
        s = fmaf(h2f(kv.k.z), qb.x, s);
        s = fmaf(h2f(kv.k.z >> 16), qb.y, s);
        s = fmaf(h2f(kv.k.w), qb.z, s);
        s = fmaf(h2f(kv.k.w >> 16), qb.w, s);
        s = group_sum<8>(s);
        const bool in = j0 + split < n;
        if (!in) s = -INFINITY;
        const float mnew = fmaxf(m, wave_max(s));  // finite: key j0 is valid
        const float r = expf(m - mnew), p = in ? expf(s - mnew) : 0.f;
        l = l * r + p;
        const uint32_t vv[4] = {in ? kv.v.x : 0u, in ? kv.v.y : 0u, in ? kv.v.z : 0u, in ? kv.v.w : 0u};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[2 * e] = fmaf(p, h2f(vv[e]), acc[2 * e] * r);
            acc[2 * e + 1] = fmaf(p, h2f(vv[e] >> 16), acc[2 * e + 1] * r);
        }
        m = mnew;
    }
    if (8 * wave < n) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = sum_splits(acc[e]);
        l = sum_splits(l);
        if (split == 0) {
            *reinterpret_cast<float4 *>(slot + 8 * sub) = make_float4(acc[0], acc[1], acc[2], acc[3]);
            *reinterpret_cast<float4 *>(slot + 8 * sub + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
            if (sub == 0) slot[64] = m, slot[65] = l;
        }
    }
}
constexpr int kResSlot = 68;  // floats per partial
__device__ __forceinline__ float attn_join(int n, int lane, const float *slots) {
    const int nw = min(kResWaves, (n + 7) / 8);
    float M = slots[64];
    #pragma unroll
    for (int w = 1; w < kResWaves; ++w) M = fmaxf(M, w < nw ? slots[w * kResSlot + 64] : M);
    float o = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < kResWaves; ++w) {
        if (w >= nw) break;
        const float e = expf(slots[w * kResSlot + 64] - M);
        l = fmaf(e, slots[w * kResSlot + 65], l);
        o = fmaf(e, slots[w * kResSlot + lane], o);
    }
    return o / l;
}

constexpr int kResBias = (5 * kResMaxD + kResMaxD + kResMaxF) / kResPlain;  // >= kResHd

struct ResLds {
    float h[kResMaxD], att[kResMaxD], catt[kResMaxD], u[kResMaxF];
    float res[64];  // a job's results on their way out
    float qkv[3 * kResHd], q2[kResHd], slots[kResWaves * kResSlot];
    float bias[kResMaxLayers][kResBias];  // this workgroup's rows: q k v | out | cross out | up | down, or cross q
    double red[2 * kResWaves];
    ResLayer layers[kResMaxLayers];
};

// the decoder's input row into xs[0, d) (plain order) by threads 0 .. d / 16 - 1
template <int ET>
__device__ __forceinline__ void embed_row(const ResArgs &a, float *xs) {
    const int k0 = 16 * int(threadIdx.x);
    if (k0 >= a.d) return;
    const float *pr = a.pos + size_t(*a.step + a.pos_base) * a.d + k0;
    float e[16];
    const uint32_t sr = a.src_row ? a.src_row[0] : kNoRow;
    if (sr != kNoRow) {
#pragma unroll
        for (int j = 0; j < 16; ++j) e[j] = a.src_emb[size_t(sr) * a.d + k0 + j];
    } else {
        dequant16<ET>(a.eq, a.es, a.ed, a.d, int(min(a.ids[0], a.elast)), k0, e);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) xs[k0 + j] = e[j] * a.emb_scale + pr[j];
}

// The gathering threads' part of a d-wide vector: values t, t + 256, ..
template <int D>
struct Gather {
    static constexpr int N = D / kResGather;
    int t;
    float x[N];  // the residual stream
    __device__ __forceinline__ Gather(int t, const float *x0) : t(t) {
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] = x0[t + k * kResGather];
    }
    __device__ __forceinline__ void vec(const float *p, float (&v)[N]) const {
        const gptr u = uniform(p);
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = ldf(u + uint32_t(4 * (t + k * kResGather)));
    }
    __device__ __forceinline__ void add(Waiter &wt, const word_t *p) {
        float v[N];
        wt.get<N>(p + t, kResGather, v);
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] += v[k];
    }
    __device__ __forceinline__ void gather(Waiter &wt, const word_t *p, float *xs) const {
        float v[N];
        wt.get<N>(p + t, kResGather, v);
#pragma unroll
        for (int k = 0; k < N; ++k) xs[pos_k4(t + k * kResGather, D / 16)] = v[k];
    }
    // LayerNorm(x) into xs: two barriers of the workgroup.  Statistics in f64 as the other step
    // kernels; d is a power of two (1 / d exact); 1 / sqrt as the hardware's estimate and a
    // Newton step in f64, then rounded to f32 (a division and a square root in f64 took 0.4 us
    // of the 0.9 a LayerNorm cost here).
    __device__ __forceinline__ void norm(const float (&g)[N], const float (&b)[N], float eps, double *red, float *xs) const {
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const double v = x[k];
            s1 += v;
            s2 += v * v;
        }
        s1 = wave_sum_f64(s1);
        s2 = wave_sum_f64(s2);
        if ((t & 63) == 0) red[2 * (t >> 6)] = s1, red[2 * (t >> 6) + 1] = s2;
        lds_barrier();
        s1 = s2 = 0.0;
#pragma unroll
        for (int k = 0; k < kResGatherWaves; ++k) s1 += red[2 * k], s2 += red[2 * k + 1];
        constexpr double inv = 1.0 / D;
        const double mean = s1 * inv, v = fmax(s2 * inv - mean * mean, 0.0) + double(eps), r0 = __builtin_amdgcn_rsq(v);
        const float rstd = float(r0 * fma(-0.5 * v * r0, r0, 1.5)), mu = float(mean);
#pragma unroll
        for (int k = 0; k < N; ++k) xs[pos_k4(t + k * kResGather, D / 16)] = (x[k] - mu) * rstd * g[k] + b[k];
        lds_barrier();
    }
};

// waves 0..7 of a head's workgroup; six barriers per layer, as head_gather
template <int T, int D>
__device__ __forceinline__ void head_dot(const ResArgs &a, ResLds &s, uint32_t tag) {
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), hd = kResHd;
    const int h = blockIdx.x, cur = int(*a.step), ns = cur + 1, nc = int(a.lens[0]);
    const int sub = lane & 7, j1 = 8 * wave + (lane >> 3);  // this lane's key of the first round
    auto load_key = [&](const __half *k, const __half *v, int j) {
        const size_t o = size_t(j) * hd + 8 * sub;
        return KeyRegs{*reinterpret_cast<const uint4 *>(k + o), *reinterpret_cast<const uint4 *>(v + o)};
    };
    auto self_k = [&](int l) { return a.kv + 2 * size_t(l) * a.self_pair + size_t(h) * a.m * hd; };
    auto cross_k = [&](int l) { return a.ckv + 2 * size_t(l) * a.cross_pair + size_t(h) * a.s * hd; };
    RowsK4<T, D == 1024 ? 8 : D == 512 ? 4 : 2, D> cq;  // the head's 64 rows of the cross q projection
    cq.load(s.layers[0].cq, h * hd, hd, wave, lane);
    // the keys of a layer's first rounds depend on nothing: requested a layer ahead
    KeyRegs sk = load_key(self_k(0), self_k(0) + a.self_pair, min(j1, a.m - 1)),
            ck = load_key(cross_k(0), cross_k(0) + a.cross_pair, min(j1, a.s - 1));
    const __half *now = reinterpret_cast<const __half *>(s.qkv + hd);  // this step's k, v
    for (int l = 0; l < a.L; ++l) {
        const Words w = words_of(a, l);
        const int ln = min(l + 1, a.L - 1);
        const __half *K = self_k(l), *V = K + a.self_pair, *CK = cross_k(l), *CV = CK + a.cross_pair;
        float *slot = s.slots + wave * kResSlot;
        cq.prepare(lane);
        lds_barrier();  // q, k, v
        auto self_key = [&](int j, KeyRegs r) {
            if (j == cur) {
                r.k = *reinterpret_cast<const uint4 *>(now + 8 * sub);
                r.v = *reinterpret_cast<const uint4 *>(now + hd + 8 * sub);
            }
            return r;
        };
        attn_partial(ns, wave, lane, s.qkv, self_key(j1, sk),
                     [&](int j) { return self_key(j, load_key(K, V, min(j, a.m - 1))); }, slot);
        lds_barrier();
        if (wave == 0) put(w.att + h * hd + lane, attn_join(ns, lane, s.slots), tag);
        sk = load_key(self_k(ln), self_k(ln) + a.self_pair, min(j1, a.m - 1));
        lds_barrier();
        lds_barrier();  // LayerNorm(x)
        cq.run(s.h, hd, wave, lane, [&](int r, float v) { s.q2[r] = v + s.bias[l][r]; });
        lds_barrier();
        attn_partial(nc, wave, lane, s.q2, ck, [&](int j) { return load_key(CK, CV, min(j, a.s - 1)); }, slot);
        lds_barrier();
        if (wave == 0) put(w.catt + h * hd + lane, attn_join(nc, lane, s.slots), tag);
        ck = load_key(cross_k(ln), cross_k(ln) + a.cross_pair, min(j1, a.s - 1));
        cq.load(s.layers[ln].cq, h * hd, hd, wave, lane);
    }
}

// waves 8..11 of a head's workgroup
template <int D>
__device__ __forceinline__ void head_gather(const ResArgs &a, ResLds &s, Waiter wt) {
    constexpr int hd = kResHd;
    const int t = int(threadIdx.x) - 64 * kResWaves, h = blockIdx.x, cur = int(*a.step);
    Gather<D> gt(t, s.u);
    float g[Gather<D>::N], b[Gather<D>::N];
    gt.vec(s.layers[0].cross_norm.g, g);
    gt.vec(s.layers[0].cross_norm.b, b);
    for (int l = 0; l < a.L; ++l) {
        const Words w = words_of(a, l);
        if (t < 3 * hd) {  // whole waves: this head's q, k, v of the step
            float v[1];
            const int part = t / hd, e = t % hd;
            wt.get<1>(w.q + part * a.d + h * hd + e, 0, v);
            if (part == 0) {
                s.qkv[t] = v[0];
            } else {  // f16 as the cache holds it
                const __half hv = __float2half(v[0]);
                a.kv[(2 * size_t(l) + part - 1) * a.self_pair + (size_t(h) * a.m + cur) * hd + e] = hv;
                reinterpret_cast<__half *>(s.qkv + hd)[(part - 1) * hd + e] = hv;
            }
        }
        lds_barrier();
        lds_barrier();
        if (l > 0) {
            const Words p = words_of(a, l - 1);
            gt.add(wt, p.cout);
            gt.add(wt, p.down);
        }
        gt.add(wt, w.out);
        gt.norm(g, b, a.eps, s.red, s.h);
        gt.vec(s.layers[min(l + 1, a.L - 1)].cross_norm.g, g);
        gt.vec(s.layers[min(l + 1, a.L - 1)].cross_norm.b, b);
        lds_barrier();
        lds_barrier();
    }
}

// waves 0..7 of a projection workgroup; twelve barriers per layer, as plain_gather
template <int T, int D>
__device__ __forceinline__ void plain_dot(const ResArgs &a, ResLds &s) {
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int g = blockIdx.x - a.H, f = a.f, ru = f / kResPlain;
    constexpr int rd = D / kResPlain, rq = 3 * rd;
    RowsK4<T, D == 1024 ? 3 : 1, D> qkv;
    RowsK4<T, 1, D> out, cout;
    RowsK4<T, D == 1024 ? 4 : D == 512 ? 2 : 1, D> up;
    RowK6 down;
    auto load_qkv = [&](const ResLayer &y) { qkv.load(y.qkv, g * rq, rq, wave, lane); };
    auto load_out = [&](const ResLayer &y) { out.load(y.out, g * rd, rd, wave, lane); };
    auto load_cout = [&](const ResLayer &y) { cout.load(y.cout, g * rd, rd, wave, lane); };
    auto load_up = [&](const ResLayer &y) { up.load(y.up, g * ru, ru, wave, lane); };
    auto load_down = [&](const ResLayer &y) { down.load(y.down, f, g * rd, rd, wave, lane); };
    load_qkv(s.layers[0]);
    load_out(s.layers[0]);
    load_cout(s.layers[0]);
    load_up(s.layers[0]);
    load_down(s.layers[0]);
    for (int l = 0; l < a.L; ++l) {
        const ResLayer &nx = s.layers[min(l + 1, a.L - 1)];
        const float *bias = s.bias[l];
        qkv.prepare(lane);
        lds_barrier();
        lds_barrier();
        qkv.run(s.h, rq, wave, lane, [&](int r, float v) { s.res[r] = v + bias[r]; });
        lds_barrier();
        load_qkv(nx);
        bias += rq;
        out.prepare(lane);
        lds_barrier();
        out.run(s.att, rd, wave, lane, [&](int r, float v) { s.res[r] = v + bias[r]; });
        lds_barrier();
        load_out(nx);
        bias += rd;
        cout.prepare(lane);
        lds_barrier();
        cout.run(s.catt, rd, wave, lane, [&](int r, float v) { s.res[r] = v + bias[r]; });
        lds_barrier();
        load_cout(nx);
        bias += rd;
        up.prepare(lane);
        lds_barrier();
        lds_barrier();
        up.run(s.h, ru, wave, lane, [&](int r, float v) { s.res[r] = fmaxf(v + bias[r], 0.f); });
        lds_barrier();
        load_up(nx);
        bias += ru;
        lds_barrier();
        if (wave < rd) {
            const float v = down.run(s.u, f, lane) + bias[wave];
            if (lane == 0) s.res[wave] = v;
        }
        lds_barrier();
        load_down(nx);
    }
}

// waves 8..11 of a projection workgroup
template <int D>
__device__ __forceinline__ void plain_gather(const ResArgs &a, ResLds &s, Waiter wt) {
    constexpr int NU = kResMaxF / kResGather;
    const int t = int(threadIdx.x) - 64 * kResWaves, f = a.f, g = blockIdx.x - a.H, ru = f / kResPlain;
    constexpr int rd = D / kResPlain, rq = 3 * rd;
    // A job's results leave in one store of whole 64-byte pieces (at d = 1024): a word stored by
    // each row's wave took 2 us longer to arrive (partial lines, written one by one).
    auto publish = [&](word_t *p, int n) {
        lds_barrier();
        if (t < n) put(p + g * n + t, s.res[t], wt.tag);
    };
    Gather<D> gt(t, s.u);
    float g1[Gather<D>::N], b1[Gather<D>::N], g2[Gather<D>::N], b2[Gather<D>::N];
    gt.vec(s.layers[0].attn_norm.g, g1);
    gt.vec(s.layers[0].attn_norm.b, b1);
    for (int l = 0; l < a.L; ++l) {
        const Words w = words_of(a, l);
        const ResLayer &ly = s.layers[l], &nx = s.layers[min(l + 1, a.L - 1)];
        if (l > 0) gt.add(wt, words_of(a, l - 1).down);
        gt.norm(g1, b1, a.eps, s.red, s.h);
        publish(w.q, rq);
        gt.vec(ly.ffn_norm.g, g2);
        gt.vec(ly.ffn_norm.b, b2);
        gt.vec(nx.attn_norm.g, g1);
        gt.vec(nx.attn_norm.b, b1);
        gt.gather(wt, w.att, s.att);
        lds_barrier();
        publish(w.out, rd);
        gt.add(wt, w.out);  // arrives while the cross attention runs
        gt.gather(wt, w.catt, s.catt);
        lds_barrier();
        publish(w.cout, rd);
        gt.add(wt, w.cout);
        gt.norm(g2, b2, a.eps, s.red, s.h);
        publish(w.u, ru);
        if (f == kResMaxF) {
            float u[NU];
            wt.get<NU>(w.u + t, kResGather, u);
#pragma unroll
            for (int k = 0; k < NU; ++k) s.u[pos_k6(t + k * kResGather, f / 64)] = u[k];
        } else {
            for (int i = t; i < f; i += kResGather) {
                float u[1];
                wt.get<1>(w.u + i, 0, u);
                s.u[pos_k6(i, f / 64)] = u[0];
            }
        }
        lds_barrier();
        publish(w.down, rd);
        if (l + 1 == a.L && t < rd) a.y[g * rd + t] = s.res[t];
    }
    if (g == 0) {
#pragma unroll
        for (int k = 0; k < Gather<D>::N; ++k) a.x_out[t + k * kResGather] = gt.x[k];
        // every workgroup has published words of this launch, so all have read the epoch
        if (t == 0) *a.epoch = wt.tag + 1;
    }
}

template <int T, int ET, int D>
__global__ __launch_bounds__(kResThreads) void k_resident(ResArgs a) {
    extern __shared__ __align__(16) unsigned char res_lds[];
    ResLds &s = *reinterpret_cast<ResLds *>(res_lds);
    const int t = threadIdx.x;
    Waiter wt{*a.epoch, a.spins, a.flag, *a.flag != 0u};
    {
        const uint32_t *src = reinterpret_cast<const uint32_t *>(a.layers);
        uint32_t *dst = reinterpret_cast<uint32_t *>(s.layers);
        for (int i = t; i < int(a.L * sizeof(ResLayer) / 4); i += kResThreads) dst[i] = src[i];
    }
    embed_row<ET>(a, s.u);  // every workgroup builds the input for itself
    __syncthreads();
    const bool head = int(blockIdx.x) < a.H;
    {  // the biases of this workgroup's rows in every layer
        const int g = int(blockIdx.x) - a.H, rd = a.d / kResPlain, ru = a.f / kResPlain, n = head ? kResHd : 6 * rd + ru;
        for (int i = t; i < a.L * n; i += kResThreads) {
            const ResLayer &y = s.layers[i / n];
            int r = i % n;
            const float *p = y.cq.bias + int(blockIdx.x) * kResHd;
            if (!head) {
                p = y.qkv.bias + 3 * rd * g;
                if (r >= 3 * rd) r -= 3 * rd, p = y.out.bias + rd * g;
                if (p == y.out.bias + rd * g && r >= rd) r -= rd, p = y.cout.bias + rd * g;
                if (p == y.cout.bias + rd * g && r >= rd) r -= rd, p = y.up.bias + ru * g;
                if (p == y.up.bias + ru * g && r >= ru) r -= ru, p = y.down.bias + rd * g;
            }
            s.bias[i / n][i % n] = p[r];
        }
    }
    __syncthreads();
    if (t < 64 * kResWaves) {
        if (head) head_dot<T, D>(a, s, wt.tag);
        else plain_dot<T, D>(a, s);
    } else {
        if (head) head_gather<D>(a, s, wt);
        else plain_gather<D>(a, s, wt);
    }
}

}  // namespace

bool step_resident_supported(int d, int f, int H, int hd, int layers, uint32_t proj, uint32_t down, uint32_t emb) {
    const bool types = (proj == GGML_Q4_K || proj == GGML_Q5_K) && down == GGML_Q6_K && emb == GGML_Q6_K;
    return types && hd == kResHd && H * hd == d && (d == 256 || d == 512 || d == kResMaxD) && f % 512 == 0 &&
           f <= kResMaxF && layers >= 1 && layers <= kResMaxLayers;
}

namespace {
template <int T>
const void *kernel_of(int d) {
    if (d == 1024) return reinterpret_cast<const void *>(&k_resident<T, GGML_Q6_K, 1024>);
    if (d == 512) return reinterpret_cast<const void *>(&k_resident<T, GGML_Q6_K, 512>);
    return reinterpret_cast<const void *>(&k_resident<T, GGML_Q6_K, 256>);
}
const void *resident_kernel(uint32_t proj, int d) {
    return proj == GGML_Q4_K ? kernel_of<GGML_Q4_K>(d) : kernel_of<GGML_Q5_K>(d);
}
hipError_t raise_lds(const void *k) {
    return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, int(sizeof(ResLds)));
}
}  // namespace

bool step_resident_fits(int d, int H, uint32_t proj, int device) {
    int cus = 0, per_cu = 0;
    const void *k = resident_kernel(proj, d);
    return hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
           raise_lds(k) == hipSuccess &&
           hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, kResThreads, sizeof(ResLds)) == hipSuccess &&
           cus * per_cu >= H + kResPlain;
}

size_t step_resident_words(int d, int f, int layers) { return size_t(layers) * (8 * d + f); }

hipError_t step_resident(const ResStep &r, hipStream_t st) {
    ResArgs a{};
    a.layers = r.layers;
    a.L = r.L;
    a.d = r.d;
    a.f = r.f;
    a.H = r.H;
    a.words = reinterpret_cast<word_t *>(r.words);
    a.epoch = r.epoch;
    a.flag = r.flag;
    a.spins = r.spins;
    a.eq = r.emb->q;
    a.es = r.emb->s;
    a.ed = r.emb->d;
    a.ids = r.ids;
    a.elast = uint32_t(r.emb->N - 1);
    a.src_emb = r.src.emb;
    a.src_row = r.src.row;
    a.pos = r.pos;
    a.pos_base = r.pos_base;
    a.emb_scale = r.emb_scale;
    a.eps = r.eps;
    a.step = r.step;
    a.lens = r.lens;
    a.kv = r.kv;
    a.ckv = r.ckv;
    a.self_pair = size_t(r.H) * r.m * kResHd;
    a.cross_pair = size_t(r.H) * r.s * kResHd;
    a.m = r.m;
    a.s = r.s;
    a.x_out = r.x_out;
    a.y = r.y;
    if (!step_resident_supported(r.d, r.f, r.H, kResHd, r.L, r.proj, GGML_Q6_K, r.emb->type)) return hipErrorInvalidValue;
    const void *k = resident_kernel(r.proj, r.d);
    void *args[] = {&a};
    return hipLaunchKernel(k, dim3(r.H + kResPlain), dim3(kResThreads), args, sizeof(ResLds), st);
}

}  // namespace mlg
