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
// workgroups: 2.0 us, so 128 share the rows).  A layer of the 600M model takes 18.1 us this
// way (q4_K, 21 keys), most of it seven hand-overs of 0.9 .. 1.5 us.
//
// Results.  Every sum has the operations and the order of the per-layer launches of k_step.hip
// (RowsK4, RowK6, Gather::norm, attn_half), so a step gives their bits, and which of the two a
// call takes shows in its time only.  Orders of its own (16 values per lane, eight waves per
// attention) took 17.4 us per layer, but then a call's tokens could differ with what other
// threads had running: a sentence of 21 ids in and 18 tokens out 7.28 (per layer) / 4.95 / 5.12 ms.
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
#include "attn_pair.hpp"
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
// instruction from whole rows of banks:
//   q4_K / q5_K rows: D / 32 lanes of one 32-value sub-block each (pos_k4);
//   q6_K rows (FFN down): K / 64 lanes of 64 values, the chunks of load_chunk<q6_K>.
template <int D>
__device__ __forceinline__ int pos_k4(int k) {
    return ((k & 31) >> 2) * (D / 8) + 4 * (k >> 5) + (k & 3);
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

constexpr int kDppPair0 = 0xA0, kDppPair1 = 0xF5;  // lane 2 i (2 i + 1) to both lanes of its pair

// v[lane] + v[lane ^ 32]
__device__ __forceinline__ float sum_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v[lane] + v[lane ^ 16]
__device__ __forceinline__ float sum_rows(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Sum over the 2^L2 chunks of a row whose value both lanes of a chunk's pair hold, in every
// lane and in group_sum's order (a mirror within twice as many lanes meets the same chunks).
template <int L2>
__device__ __forceinline__ float sum_chunks(float v) {
    if constexpr (L2 >= 1) v += dpp_mov<kDppXor2>(v);
    if constexpr (L2 >= 2) v += dpp_mov<kDppHalfMirror>(v);
    if constexpr (L2 >= 3) v += dpp_mov<kDppMirror>(v);
    if constexpr (L2 >= 4) v = sum_rows(v);
    return v;
}

// Rows of a q4_K / q5_K matrix, NP passes of 8 RPW rows: D / 32 lanes per row, one 32-value
// sub-block each, RPW rows per wave.  The two lanes of a 64-value chunk hold 16 of its 32
// packed bytes each and read the other's by DPP; lane 2 c sums the low nibbles, lane 2 c + 1
// the high ones, and both form the chunk's value (k4_chunk).  Every sum has the operations and
// the order of dot_chunk and group_sum, one chunk per lane.
template <int T, int NP, int D>
struct RowsK4 {
    static constexpr int LPR = D / 32, RPW = 64 / LPR, L2 = D == 1024 ? 4 : D == 512 ? 3 : 2;
    static constexpr int B = T == GGML_Q4_K ? 144 : 176;
    uint4 h[NP], q[NP], qh[T == GGML_Q5_K ? NP : 1];  // qh: q5_K's fifth bits
    __device__ __forceinline__ static int row(int p, int wave, int lane) { return (p * kResWaves + wave) * RPW + lane / LPR; }
    __device__ __forceinline__ void load(const ResMat &mt, int row0, int rows, int wave, int lane) {
        __builtin_amdgcn_sched_barrier(0);  // the registers' last values have been used
        // q5_K: the offsets are formed again each time (kept over the layers, they spill)
        if constexpr (T == GGML_Q5_K) asm volatile("" : "+v"(lane));
        const int sb = lane & (LPR - 1), hi = sb & 1, g = (sb >> 1) & 3;
        constexpr int rb = (D >> 8) * B;
        const gptr m0 = uniform(mt.q) + size_t(row0) * rb;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const uint32_t off = uint32_t(min(row(p, wave, lane), rows - 1) * rb + (sb >> 3) * B);
            h[p] = ld16(m0 + off);
            q[p] = ld16(m0 + (off + (B - 128) + 32 * g + 16 * hi));
            if constexpr (T == GGML_Q5_K) qh[p] = ld16(m0 + (off + 16 + 16 * hi));
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // h.y becomes the chunk's 6-bit (scale, min) pairs (sc0, m0, sc1, m1), a byte each.  Done
    // while the wave has nothing to wait for but its vector.
    __device__ __forceinline__ void prepare(int lane) {
        const int g = ((lane & (LPR - 1)) >> 1) & 3, sh0 = 8 * ((2 * g) & 3);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const uint32_t B0 = h[p].y >> sh0, B1 = h[p].z >> sh0, B2 = h[p].w >> sh0;
            // two bytes each: the pair's scales and mins
            const uint32_t sc = g >= 2 ? ((B2 & 0x0F0Fu) | ((B0 >> 2) & 0x3030u)) : (B0 & 0x3F3Fu);
            const uint32_t mn = g >= 2 ? (((B2 >> 4) & 0x0F0Fu) | ((B1 >> 2) & 0x3030u)) : (B1 & 0x3F3Fu);
            h[p].y = __builtin_amdgcn_perm(mn, sc, 0x05010400u);
        }
        // here, not where the values are used (behind the barrier)
#pragma unroll
        for (int p = 0; p < NP; ++p) asm volatile("" : "+v"(h[p].x), "+v"(h[p].y));
    }
    // the chunk's value of every pass
    __device__ __forceinline__ void chunks(const float *xs, int lane, float (&v)[NP]) const {
        const int sb = lane & (LPR - 1), hi = sb & 1, g = (sb >> 1) & 3;
        const uint32_t mask = hi ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
        float a[NP], s = 0.f;
#pragma unroll
        for (int p = 0; p < NP; ++p) a[p] = 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float4 xv = *reinterpret_cast<const float4 *>(xs + u * (D / 8) + 4 * sb);
            const float x[4] = {xv.x, xv.y, xv.z, xv.w};
            s += x[0], s += x[1], s += x[2], s += x[3];
            uint32_t w[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const uint32_t wo = (&q[p].x)[u & 3];
                w[p] = u < 4 ? dpp_mov<kDppPair0>(wo) : dpp_mov<kDppPair1>(wo);
                if constexpr (T == GGML_Q4_K) {
                    w[p] &= mask;  // high: 16 * nibble, scaled back below
                } else {
                    const uint32_t ho = (&qh[p].x)[u & 3], hb = u < 4 ? dpp_mov<kDppPair0>(ho) : dpp_mov<kDppPair1>(ho);
                    w[p] = ((w[p] >> (4 * hi)) & 0x0F0F0F0Fu) | (((hb >> (2 * g + hi)) & 0x01010101u) << 4);
                }
            }
            dot4u8_items(w, x, a);
        }
        const float s0 = dpp_mov<kDppPair0>(s), s1 = dpp_mov<kDppPair1>(s);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            if constexpr (T == GGML_Q4_K) a[p] *= hi ? 0.0625f : 1.f;
            const uint32_t sm = h[p].y;
            v[p] = k4_chunk(0.f, h2f(h[p].x), h2f(h[p].x >> 16), ub0(sm), ub1(sm), ub2(sm), ub3(sm),
                            dpp_mov<kDppPair0>(a[p]), dpp_mov<kDppPair1>(a[p]), s0, s1);
        }
    }
    // store(row of the job, sum) by the first lane of each row
    template <class F>
    __device__ __forceinline__ void run(const float *xs, int rows, int wave, int lane, F &&store) const {
        float v[NP];
        chunks(xs, lane, v);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const float r = sum_chunks<L2>(v[p]);
            const int at = row(p, wave, lane);
            if ((lane & (LPR - 1)) == 0 && at < rows) store(at, r);
        }
    }
    // the out-projections: a row's sums over the chunks of each head group of step_attn_head
    // (head_geometry: D / 64 heads of one chunk in at most 8 groups) to out[row 8 + group]
    static constexpr int GL2 = D == 1024 ? 1 : 0, kParts = (D / 64) >> GL2;
    static_assert(kParts <= 8, "a row's partial sums take 8 floats");
    __device__ __forceinline__ void run_parts(const float *xs, int rows, int wave, int lane, float *out) const {
        static_assert(NP == 1, "one pass");
        float v[1];
        chunks(xs, lane, v);
        const float r = sum_chunks<GL2>(v[0]);
        const int at = row(0, wave, lane), sb = lane & (LPR - 1);
        if ((sb & ((2 << GL2) - 1)) == 0 && at < rows) out[8 * at + (sb >> (1 + GL2))] = r;
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
            for (int k = 0; k < 4; ++k) {  // sums in the order of gemv_load_x and dot_chunk
                const float4 v = *reinterpret_cast<const float4 *>(xs + 4 * lanes * (4 * k + u) + o);
                const float x[4] = {v.x, v.y, v.z, v.w};
                q[k] = dot4u8(w4[k], x, q[k]);
                sx[k] += x[0], sx[k] += x[1], sx[k] += x[2], sx[k] += x[3];
            }
        }
        float acc = q6_chunk(0.f, h2f(w.c.x), sc, q, sx);
        if (lane >= lanes) acc = 0.f;
        acc = sum_rows(group_sum<16>(acc));
        return sum_halves(acc);
    }
};

constexpr int kResBias = (5 * kResMaxD + kResMaxD + kResMaxF) / kResPlain;  // >= kResHd

struct ResLds {
    float h[kResMaxD], att[kResMaxD], catt[kResMaxD], u[kResMaxF];
    float res[64];  // a job's results on their way out
    float qkv[3 * kResHd], q2[kResHd];
    float wsc[2 * 512], slots[2 * kHalfSlot];  // of the two waves of an attention (attn_half)
    float bias[kResMaxLayers][kResBias];  // this workgroup's rows: q k v | out | cross out | up | down, or cross q
    double red[2 * kResWaves];
    ResLayer layers[kResMaxLayers];
};

static_assert(sizeof(ResLds) <= 64 * 1024, "more needs the kernel's LDS limit raised");

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

// float(1 / sqrt(v)) as the other step kernels round it: a correctly rounded square root and a
// correctly rounded division in f64, then to f32.  Those two take 0.4 of the 0.9 us that a
// LayerNorm would cost here, so: the hardware's estimate (2^-24) and a Newton step, whose
// 2^-40 decides the rounding to f32 in all but one of some 10^4 cases.
__device__ __forceinline__ float ln_rstd(double v) {
    const double r0 = __builtin_amdgcn_rsq(v), r = r0 * fma(-0.5 * v * r0, r0, 1.5);
    const float lo = float(r * (1.0 - 0x1p-40)), hi = float(r * (1.0 + 0x1p-40));
    return lo == hi ? lo : float(1.0 / sqrt(v));
}

// The gathering threads' part of a D-wide vector: values at(0 .. 3) of the threads t < D / 4
// (whole waves; a wave's 256 values in 64-value runs, as they are polled).
template <int D>
struct Gather {
    static constexpr int N = 4;
    int t;
    bool on;  // wave-uniform
    float x[N];  // the residual stream
    __device__ __forceinline__ int at(int k) const { return 4 * (t & ~63) + 64 * k + (t & 63); }
    __device__ __forceinline__ Gather(int t, const float *x0) : t(t), on(t < D / 4) {
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] = x0[on ? at(k) : 0];
    }
    // values 4 t .. 4 t + 3
    __device__ __forceinline__ float4 vec(const float *p) const {
        const u32x4_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t *>(
            uniform(p) + uint32_t(on ? 16 * t : 0));
        return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    }
    __device__ __forceinline__ void add(Waiter &wt, const word_t *p) {
        if (!on) return;
        float v[N];
        wt.get<N>(p + at(0), 64, v);
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] += v[k];
    }
    __device__ __forceinline__ void gather(Waiter &wt, const word_t *p, float *xs) const {
        if (!on) return;
        float v[N];
        wt.get<N>(p + at(0), 64, v);
#pragma unroll
        for (int k = 0; k < N; ++k) xs[pos_k4<D>(at(k))] = v[k];
    }
    // LayerNorm(x) into xs: two barriers of the workgroup.  Statistics in f64 with the sums and
    // the order of ln_to_lds (thread t sums values 4 t .. 4 t + 3, which it reads back from xs,
    // then the wave, then the waves); D is a power of two, so 1 / D is exact.
    __device__ __forceinline__ void norm(const float4 &g, const float4 &b, float eps, double *red, float *xs) const {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        double s1 = 0.0, s2 = 0.0;
        if (on) {
#pragma unroll
            for (int k = 0; k < N; ++k) xs[at(k)] = x[k];
            __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's LDS writes are done
            __builtin_amdgcn_wave_barrier();
            v = ld4(xs, t);
            ln_acc(v, s1, s2);
        }
        s1 = wave_sum_f64(s1);
        s2 = wave_sum_f64(s2);
        if ((t & 63) == 0) red[t >> 6] = s1, red[kResGatherWaves + (t >> 6)] = s2;
        lds_barrier();
        s1 = (red[0] + red[1]) + (red[2] + red[3]);
        s2 = (red[4] + red[5]) + (red[6] + red[7]);
        constexpr double inv = 1.0 / D;
        const double mean = s1 * inv, ms = s2 * inv, var = fmax(fma(-mean, mean, ms), 0.0);
        const float rstd = ln_rstd(var + double(eps)), mu = float(mean);
        if (on) *reinterpret_cast<float4 *>(xs + pos_k4<D>(4 * t)) = ln_apply(v, mu, rstd, g, b);
        lds_barrier();
    }
};
static_assert(kResMaxF == 16 * kResGather, "plain_gather's largest poll");
static_assert(kResGatherWaves == 4, "norm adds four waves' sums");

// waves 0..7 of a head's workgroup; six barriers per layer, as head_gather
template <int T, int D>
__device__ __forceinline__ void head_dot(const ResArgs &a, ResLds &s, uint32_t tag) {
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), hd = kResHd;
    const int h = blockIdx.x, cur = int(*a.step), ns = cur + 1, nc = int(a.lens[0]);
    const int sub = lane & 7, split = lane >> 3;
    // waves 0, 1 attend to the self cache, waves 2, 3 to the cross K/V (attn_half's two waves):
    // each keeps one attention's first chunk, requested a layer ahead (it depends on nothing)
    const bool self = wave < 2, cross = wave == 2 || wave == 3;
    const int q = wave & 1;
    uint4 kr[kHalfU], vr[kHalfU];
    auto load_keys = [&](int l, int c) {
        const int L = self ? a.m : a.s;
        const __half *k = self ? a.kv + 2 * size_t(l) * a.self_pair + size_t(h) * a.m * hd
                               : a.ckv + 2 * size_t(l) * a.cross_pair + size_t(h) * a.s * hd;
        const gptr K = uniform(k), V = uniform(k + (self ? a.self_pair : a.cross_pair));
#pragma unroll
        for (int u = 0; u < kHalfU; ++u) {
            const uint32_t o = uint32_t(min(half_key(8, c, u, q) + split, L - 1)) * uint32_t(2 * hd) + uint32_t(16 * sub);
            kr[u] = ld16(K + o);
            vr[u] = ld16(V + o);
        }
    };
    RowsK4<T, D == 1024 ? 4 : D == 512 ? 2 : 1, D> cq;  // the head's 64 rows of the cross q projection
    cq.load(s.layers[0].cq, h * hd, hd, wave, lane);
    if (self || cross) load_keys(0, 0);
    const __half *now = reinterpret_cast<const __half *>(s.qkv + hd);  // this step's k, v
    float *wsc = s.wsc + q * 512, *slot = s.slots + q * kHalfSlot;
    auto attend = [&](int l, int n, const float *qv, auto &&fix) {
        const float4 qa = *reinterpret_cast<const float4 *>(qv + 8 * sub), qb = *reinterpret_cast<const float4 *>(qv + 8 * sub + 4);
        fix(0);
        attn_half<kResHd>(n, q, qa, qb, kr, vr, [&](int c) {
            load_keys(l, c);
            fix(c);
        }, wsc, slot);
    };
    auto publish = [&](word_t *p) {
        attn_combine2<kResHd>(s.slots, s.slots + kHalfSlot, s.res);
        put(p + h * hd + lane, s.res[lane], tag);
    };
    for (int l = 0; l < a.L; ++l) {
        const Words w = words_of(a, l);
        const int ln = min(l + 1, a.L - 1);
        cq.prepare(lane);
        lds_barrier();  // q, k, v
        if (self)
            attend(l, ns, s.qkv, [&](int c) {
                // the cache's slot of this step is being written: its key comes from LDS
#pragma unroll
                for (int u = 0; u < kHalfU; ++u)
                    if (half_key(8, c, u, q) + split == cur) {
                        kr[u] = *reinterpret_cast<const uint4 *>(now + 8 * sub);
                        vr[u] = *reinterpret_cast<const uint4 *>(now + hd + 8 * sub);
                    }
            });
        lds_barrier();
        if (wave == 0) publish(w.att);
        if (self) load_keys(ln, 0);
        lds_barrier();
        lds_barrier();  // LayerNorm(x)
        cq.run(s.h, hd, wave, lane, [&](int r, float v) { s.q2[r] = v + s.bias[l][r]; });
        lds_barrier();
        if (cross) attend(l, nc, s.q2, [](int) {});
        lds_barrier();
        if (wave == 2) publish(w.catt);
        if (cross) load_keys(ln, 0);
        cq.load(s.layers[ln].cq, h * hd, hd, wave, lane);
    }
}

// waves 8..11 of a head's workgroup
template <int D>
__device__ __forceinline__ void head_gather(const ResArgs &a, ResLds &s, Waiter wt) {
    constexpr int hd = kResHd;
    const int t = int(threadIdx.x) - 64 * kResWaves, h = blockIdx.x, cur = int(*a.step);
    Gather<D> gt(t, s.u);
    float4 g = gt.vec(s.layers[0].cross_norm.g), b = gt.vec(s.layers[0].cross_norm.b);
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
        g = gt.vec(s.layers[min(l + 1, a.L - 1)].cross_norm.g);
        b = gt.vec(s.layers[min(l + 1, a.L - 1)].cross_norm.b);
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
    RowsK4<T, D == 1024 ? 2 : 1, D> qkv;
    RowsK4<T, 1, D> out, cout;
    RowsK4<T, D == 1024 ? 2 : 1, D> up;
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
        out.prepare(lane);
        lds_barrier();
        out.run_parts(s.att, rd, wave, lane, s.res);
        lds_barrier();
        load_out(nx);
        cout.prepare(lane);
        lds_barrier();
        cout.run_parts(s.catt, rd, wave, lane, s.res);
        lds_barrier();
        load_cout(nx);
        bias += rq + 2 * rd;
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
template <int T, int D>
__device__ __forceinline__ void plain_gather(const ResArgs &a, ResLds &s, Waiter wt) {
    const int t = int(threadIdx.x) - 64 * kResWaves, f = a.f, g = blockIdx.x - a.H, ru = f / kResPlain;
    constexpr int rd = D / kResPlain, rq = 3 * rd;
    // A job's results leave in one store of whole 64-byte pieces (at d = 1024): a word stored by
    // each row's wave took 2 us longer to arrive (partial lines, written one by one).
    auto publish = [&](word_t *p, int n) {
        lds_barrier();
        if (t < n) put(p + g * n + t, s.res[t], wt.tag);
    };
    // the same for an out-projection, whose rows are sums over the head groups in order
    auto publish_parts = [&](word_t *p, const float *bias) {
        lds_barrier();
        if (t < rd) {
            const float *r = s.res + 8 * t;
            float v = r[0];
#pragma unroll
            for (int k = 1; k < RowsK4<T, 1, D>::kParts; ++k) v += r[k];
            put(p + g * rd + t, v + bias[t], wt.tag);
        }
    };
    // words i, i + 256, .. of the FFN's hidden vector, n of them at once
    auto gather_u = [&](auto nc, const word_t *p, int &i) {
        constexpr int n = decltype(nc)::value;
        float u[n];
        wt.get<n>(p + i, kResGather, u);
#pragma unroll
        for (int k = 0; k < n; ++k) s.u[pos_k6(i + k * kResGather, f / 64)] = u[k];
        i += n * kResGather;
    };
    Gather<D> gt(t, s.u);
    float4 g1 = gt.vec(s.layers[0].attn_norm.g), b1 = gt.vec(s.layers[0].attn_norm.b), g2, b2;
    for (int l = 0; l < a.L; ++l) {
        const Words w = words_of(a, l);
        const ResLayer &ly = s.layers[l], &nx = s.layers[min(l + 1, a.L - 1)];
        if (l > 0) gt.add(wt, words_of(a, l - 1).down);
        gt.norm(g1, b1, a.eps, s.red, s.h);
        publish(w.q, rq);
        g2 = gt.vec(ly.ffn_norm.g);
        b2 = gt.vec(ly.ffn_norm.b);
        g1 = gt.vec(nx.attn_norm.g);
        b1 = gt.vec(nx.attn_norm.b);
        gt.gather(wt, w.att, s.att);
        lds_barrier();
        publish_parts(w.out, s.bias[l] + rq);
        gt.add(wt, w.out);  // arrives while the cross attention runs
        gt.gather(wt, w.catt, s.catt);
        lds_barrier();
        publish_parts(w.cout, s.bias[l] + rq + rd);
        gt.add(wt, w.cout);
        gt.norm(g2, b2, a.eps, s.red, s.h);
        publish(w.u, ru);
        // f / 256 words per thread, whole powers of two polled at once (f is a multiple of 512):
        // one by one, a step of six layers of FFN 2560 took 152 us, now 136 (3584: 161, 139)
        int i = t;
        static_for<0, 4>([&](auto jc) {
            constexpr int n = 16 >> decltype(jc)::value;
            if (f & (n * kResGather)) gather_u(std::integral_constant<int, n>{}, w.u, i);
        });
        lds_barrier();
        publish(w.down, rd);
        if (l + 1 == a.L && t < rd) a.y[g * rd + t] = s.res[t];
    }
    if (g == 0) {
#pragma unroll
        for (int k = 0; k < Gather<D>::N; ++k)
            if (gt.on) a.x_out[gt.at(k)] = gt.x[k];
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
        else plain_gather<T, D>(a, s, wt);
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
}  // namespace

bool step_resident_fits(int d, int H, uint32_t proj, int device) {
    int cus = 0, per_cu = 0;
    const void *k = resident_kernel(proj, d);
    return hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
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
