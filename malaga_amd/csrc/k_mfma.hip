// Dequant GEMM on the MFMA units (src/model.rs:463-477 encoder prefill, and the
// projections of decode batches too large for the register GEMV):
//   Y[m][n] = sum_k X[m][k] W[n][k] + bias[n] (+ R[m][n]) (relu)
//
// Exactness: the integer quants (q4_K / q5_K nibbles, q6_K 6-bit values - 32,
// q8_0 int8) are exact in f16, so the MFMA multiplies them by X, which is split
// into two f16 terms x = hi + lo (|x - hi - lo| <= 2^-22 |x|), with f32
// accumulation.  The block scales go where they cost least VALU work (block_mfma):
// q4_K / q5_K fold the 6-bit sub-block scale into B (a q, exact in f16), q6_K its int8
// group scale as the exact pair bh + bl = q sc (MW<q6_K>::b_split), so that a
// super-block's 8 slices of 32 chain in the 16x16x32 MFMA's C operand and d is applied
// once per block; the k-quant mins are one more MFMA per block over the 8 sub-block
// averages of x; q8_0 applies its scale per slice of 32 in f32.
//
// Tiling: a workgroup of 4 or 8 waves owns BM rows of X and 16 or 32 rows of W per wave
// (tile_of).  K is consumed in steps of 256 (one k-quant super-block): the X step is staged
// in LDS as hi/lo f16 (plus the sub-block averages for the formats with mins), while the
// next step's X and W are in flight in registers.  Each wave keeps its W rows in registers
// in the MFMA B-operand layout (lane l: row l % 16, k-group l / 16) and reads A (X) from LDS.
// f16 MFMA operand conversion of quant bytes uses v_perm (byte -> 0x64xx = 1024 +
// byte) and one packed f16 subtraction.
#include "kernels.hpp"
#include "mfma_core.hpp"

#include <algorithm>

namespace mlg {

namespace {

// LDS row stride of the staged X (halves).  272 (136 dwords): the A-fragment reads and the
// 16-byte staging stores have no bank conflicts (rocprofv3: 264 and 280 left 49-65 K conflict
// cycles per CU in each encoder GEMM launch, 272 none for q6_K).  The resident-X LM head
// (k_mfma_rx) uses the same 8-mod-64-dword stride (rx_stride); k_drx keeps K + 8 (its bank
// conflicts are off the critical path)
constexpr int kXS = kStep + 16;
constexpr int kXM = 32;  // halves per row of the sub-block averages (XStage::store)

// X staging of one 256-wide K step into LDS as f16 hi / lo (+ the sub-block averages for
// the formats with mins).  Each thread converts chunks of 8 values and writes them as one
// 16-byte store; 16 consecutive lanes take 16 consecutive chunks of one row, so each
// store of 16 lanes covers 256 contiguous bytes of LDS (no bank conflicts).  Thread t:
// rows t / 16 + (NTH / 16) u, chunks t % 16 + 16 h (32 chunks per row and step).
// Chunk c holds x[8 c .. 8 c + 7], or for split-B types the two 4-value groups that
// split_pos puts there: x[32 (c / 4) + 4 (c % 4) + e] and x[32 (c / 4) + 16 + 4 (c % 4) + e].
template <int BM, int NTH, bool SPLIT>
struct XStage {
    static constexpr int R = NTH / 16, RP = BM / R;  // rows per pass, row passes
    static_assert(RP >= 1 && BM % R == 0, "X tile / thread count");
    float4 v[RP][2][2];  // [row pass][chunk h][half]
    // a scalar base and a 32-bit lane offset per row (rows past M read row M - 1: their
    // products are not stored), so that a load needs no vector address arithmetic
    const char *base;
    uint32_t off[RP];
    int cl, rg;
    __device__ void init(const float *x, int ldx, int m0, int M, int t) {
        cl = t & 15, rg = t >> 4;
        base = reinterpret_cast<const char *>(x + size_t(m0) * ldx);
#pragma unroll
        for (int u = 0; u < RP; ++u)
            off[u] = (uint32_t(min(rg + R * u, M - 1 - m0)) * uint32_t(ldx) + uint32_t(koff(cl, 0))) * 4u;
    }
    __device__ static int koff(int c, int half) {
        if constexpr (SPLIT) return 32 * (c >> 2) + 16 * half + 4 * (c & 3);
        else return 8 * c + 4 * half;
    }
    __device__ void load(int kb) {
        const char *p = base + size_t(kb) * (kStep * 4);
#pragma unroll
        for (int u = 0; u < RP; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    v[u][h][f] = *reinterpret_cast<const float4 *>(p + off[u] + 4 * (koff(16 * h, f) - koff(0, 0)));
    }
    // xm (SUMS): per row the 8 sub-block averages of the step as the A operand of the min
    // term (block_mfma), kXM halves: [hi of sub-blocks 0..7 | 2048 lo of 0..7 | zeros]
    template <bool SUMS>
    __device__ void store(_Float16 *xh, _Float16 *xl, _Float16 *xm) const {
        float sums[RP * 2];
#pragma unroll
        for (int u = 0; u < RP; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int m = rg + R * u, c = cl + 16 * h;
                const float e[8] = {v[u][h][0].x, v[u][h][0].y, v[u][h][0].z, v[u][h][0].w,
                                    v[u][h][1].x, v[u][h][1].y, v[u][h][1].z, v[u][h][1].w};
                h8_t hv, lv;
                split_h8(e, hv, lv);
                *reinterpret_cast<h8_t *>(xh + m * kXS + 8 * c) = hv;
                *reinterpret_cast<h8_t *>(xl + m * kXS + 8 * c) = lv;
                if constexpr (SUMS) {  // sums of 32: this chunk and the next three (a quad of lanes)
                    float sm = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
                    sm += dpp_mov<kDppXor1>(sm);
                    sums[2 * u + h] = sm + dpp_mov<kDppXor2>(sm);
                }
            }
        if constexpr (SUMS) {  // lane i of a quad splits and stores the quad's sums i, i + 4, ..
#pragma unroll
            for (int k = 0; k < (2 * RP + 3) / 4; ++k) {
                const int i = 4 * k + (cl & 3);
                float sm = sums[4 * k];
#pragma unroll
                for (int e = 1; e < 4; ++e)
                    if (4 * k + e < 2 * RP) sm = i == 4 * k + e ? sums[4 * k + e] : sm;
                sm *= 1.f / 32;  // an average is in the f16 range wherever its values are
                const _Float16 ah = _Float16(sm), al = _Float16((sm - float(ah)) * 2048.f);
                _Float16 *p = xm + (rg + R * (i >> 1)) * kXM + (cl >> 2) + 4 * (i & 1);
                if (2 * RP % 4 == 0 || i < 2 * RP) p[0] = ah, p[8] = al;
            }
        }
    }
    // the zero half of the xm rows (before the first store; a barrier follows)
    __device__ static void clear_sums(_Float16 *xm, int t) {
        for (int i = t; i < BM * 2; i += NTH)
            *reinterpret_cast<uint4 *>(xm + (i >> 1) * kXM + 16 + 8 * (i & 1)) = make_uint4(0, 0, 0, 0);
    }
};

struct MfmaArgs {
    WPtr w;
    const float *x;
    int ldx, M;
    float *y;
    int ldy;
    const float *bias, *R;
    int ldr, relu;
    float *part;  // split K: raw sums [gridDim.z][M][N], epilogue in k_splitk_reduce
    int mask_id;  // MODE 1: row index never selected (-1: none)
    float *pv;    // MODE 1: argmax partials [M][parts], one per workgroup
    uint32_t *pi;
    int parts;
};


// acc[j][mt] += one 256-wide K block of W tiles cur[j] (16 rows each, B operand) with the
// staged X rows (A operand).  Bound by VALU work beside the MFMAs, so the scales stay out of
// the slices:
//   FOLD (q4_K / q5_K): B = a_s (q - z), z the middle of the quant range, the block's slices
//     chain in C; what is left of the mins, sum_s T_s sum_s x with T_s = z d a_s - dmin m_s, is
//     one MFMA per tile and block over the averages of x (hi | 2048 lo | hi): per block
//     acc += d C + 32 T.  Neither C nor T carries the mean of the weights, which cancels
//     (off 64 bits, x of zero mean / after ReLU: scales and mins per slice in f32 3.0e-7 /
//     5.4e-7, uncentred 5.0e-7, centred with separate sums of a_s x and m_s x 2.0e-7 / 9.1e-7).
//   SPLIT (q6_K): B = bh + bl, three MFMAs per slice, d once per block.
//   q8_0, f16: the slice's scale (1) in f32 (chained in acc, f16 would round twice per slice:
//     1.6e-7 off 64 bits instead of 1.1e-7).
// A fragments of slice s + 1 are read from LDS while slice s runs on the MFMA.
template <int T, int MT, int WT>
__device__ __forceinline__ void block_mfma(const typename MW<T>::Regs (&cur)[WT], const _Float16 *xh,
                                           const _Float16 *xl, const _Float16 *xm, int ln, int kq,
                                           f4_t (&acc)[WT][MT]) {
    using W = MW<T>;
    constexpr f4_t zero = {0.f, 0.f, 0.f, 0.f};
    h8_t ahs[2][MT], als[2][MT];
    auto read_a = [&](int s, h8_t (&ah)[MT], h8_t (&al)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int xo = (mt * 16 + ln) * kXS + 32 * s + 8 * kq;
            ah[mt] = *reinterpret_cast<const h8_t *>(xh + xo);
            al[mt] = *reinterpret_cast<const h8_t *>(xl + xo);
        }
    };
    read_a(0, ahs[0], als[0]);
    [[maybe_unused]] f4_t cb[WT][MT];
    [[maybe_unused]] FoldPrep fp[WT];
    if constexpr (W::FOLD) {
#pragma unroll
        for (int j = 0; j < WT; ++j) fp[j] = fold_prep<W, W::MID_NA>(cur[j]);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        if (s + 1 < 8) read_a(s + 1, ahs[(s + 1) & 1], als[(s + 1) & 1]);
        if constexpr (W::FOLD || W::SPLIT) {
            h8_t bh[WT], bl[WT];
#pragma unroll
            for (int j = 0; j < WT; ++j) {
                if constexpr (W::FOLD) bh[j] = W::b_fold_mid(cur[j], fp[j], s);
                else W::b_split(cur[j], s, bh[j], bl[j]);
            }
            if constexpr (W::SPLIT) {  // tile by tile: a fragment of A is done with after its three products
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const h8_t ah = ahs[s & 1][mt], al = als[s & 1][mt];
#pragma unroll
                    for (int j = 0; j < WT; ++j)
                        cb[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bh[j], s ? cb[j][mt] : zero, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < WT; ++j) cb[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh[j], cb[j][mt], 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < WT; ++j) cb[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl[j], cb[j][mt], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int j = 0; j < WT; ++j)
                        cb[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahs[s & 1][mt], bh[j], s ? cb[j][mt] : zero, 0, 0, 0);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int j = 0; j < WT; ++j)
                        cb[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(als[s & 1][mt], bh[j], cb[j][mt], 0, 0, 0);
            }
        } else {
            float sc[WT], mn[WT];
            h8_t bop[WT];
#pragma unroll
            for (int j = 0; j < WT; ++j) {
                W::scale(cur[j], s, sc[j], mn[j]);
                bop[j] = W::b(cur[j], s);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const h8_t ah = ahs[s & 1][mt], al = als[s & 1][mt];
#pragma unroll
                for (int j = 0; j < WT; ++j) {
                    f4_t tmp = zero;
                    tmp = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bop[j], tmp, 0, 0, 0);
                    tmp = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bop[j], tmp, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[j][mt][r] = fmaf(sc[j], tmp[r], acc[j][mt][r]);
                }
            }
        }
    }
    if constexpr (W::FOLD) {
        // T_s = z d a_s - dmin m_s, what is left of the mins, as an f16 pair: exact products and
        // one rounding in f32, scaled by 64 / p (p: the power of two below the larger of z d and
        // dmin) so that |T| <= 16128 and T / 2048 stays normal.  k-groups of the MFMA: Thi with
        // the averages' hi, Thi / 2048 with 2048 lo, Tlo with hi again, zeros.
        h8_t bt[WT];
        float d[WT], back[WT];
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            d[j] = h2f(cur[j].hdr.x);
            const float dmin = h2f(cur[j].hdr.x >> 16), zd = float(W::MID) * d[j];
            const uint32_t pb = __float_as_uint(fmaxf(fmaxf(fabsf(zd), fabsf(dmin)), 1e-30f)) & 0x7f800000u;
            const float inv = __uint_as_float(0x7f000000u - pb) * 64.f, da = zd * inv, dm = dmin * inv;
            back[j] = 0.5f * __uint_as_float(pb);  // 32 p / 64
            float t[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const h2_t av = __builtin_bit_cast(h2_t, fp[j].a[s >> 1]), mv = __builtin_bit_cast(h2_t, fp[j].m[s >> 1]);
                t[s] = fmaf(da, float(av[s & 1]), -(dm * float(mv[s & 1])));
            }
            h8_t hi, lo;
            split_h8(t, hi, lo);
            const _Float16 f = kq == 1 ? _Float16(1.f / 2048) : _Float16(1.f);
            const h8_t f8 = {f, f, f, f, f, f, f, f};
            bt[j] = kq < 2 ? hi * f8 : lo;
        }
        const int ao = kq == 1 ? 8 : kq == 3 ? 16 : 0;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const h8_t am = *reinterpret_cast<const h8_t *>(xm + (mt * 16 + ln) * kXM + ao);
#pragma unroll
            for (int j = 0; j < WT; ++j) {
                const f4_t tb = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, bt[j], zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[j][mt][r] = fmaf(back[j], tb[r], fmaf(d[j], cb[j][mt][r], acc[j][mt][r]));
            }
        }
    } else if constexpr (W::SPLIT) {
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            const float d = W::d_of(cur[j]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[j][mt][r] = fmaf(d, cb[j][mt][r], acc[j][mt][r]);
        }
    }
}

// y[m][n] = sum_{z < ks} part[z][m][n] (in order) + bias[n] (+ R[m][n]) (relu)
__global__ __launch_bounds__(256) void k_splitk_reduce(const float *part, int ks, int M, int N, const float *bias,
                                                        const float *R, int ldr, int relu, float *y, int ldy) {
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x, mn = size_t(M) * N;
    if (i >= mn) return;
    const int m = int(i / N), n = int(i % N);
    float v = 0.f;
    for (int z0 = 0; z0 < ks; z0 += 8) {
        float p8[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p8[u] = z0 + u < ks ? part[size_t(z0 + u) * mn + i] : 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (z0 + u < ks) v = (z0 + u == 0) ? p8[u] : v + p8[u];
    }
    if (bias) v += bias[n];
    if (R) v += R[size_t(m) * ldr + n];
    if (relu) v = fmaxf(v, 0.f);
    y[size_t(m) * ldy + n] = v;
}

// ------------------------------------------------------------- tile kernel
//
// NW waves, each owning WT 16-row tiles of W: a workgroup covers 16 NW WT rows of W and BM
// rows of X, and one staging of X per K step serves all its waves.  A wave reads each X
// fragment from LDS once per slice and uses it for its WT tiles.
template <int BM>
constexpr size_t mfma_lds() {
    return (size_t(2) * BM * kXS + size_t(BM) * kXM) * sizeof(_Float16);
}

// MODE 0 stores Y (or split-K partials); MODE 1 (the greedy LM head of 33..64 rows) keeps
// a (value, lowest index) argmax per X row and workgroup instead (gridDim.y = z = 1).
// TL: W from the tile-major copy a.w.t (q6_K / q4_K).
// Waves per SIMD that the kernel is scheduled for: what its LDS leaves room for.  It is
// dynamic, so the compiler cannot see that, and for the 3 or 4 that its registers would
// allow it kept the reads of A close to their use (q6_K 1024 x 4096 at 2048 rows 65.9 ->
// 65.2 us, q8_0 2048 x 2048 at 512 rows 29.6 -> 27.1, q4_K 3072 x 1024 at 911 25.5 -> 24.9).
constexpr int mfma_waves(int bm) { return bm == 64 ? 2 : 4; }
template <int T, int BM, int NW, int WT, bool TL, int MODE = 0>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(mfma_waves(BM), mfma_waves(BM)))) void k_mfma(
    MfmaArgs a) {
    using W = MW<T>;
    constexpr int MT = BM / 16;
    constexpr int NTH = NW * 64;
    extern __shared__ __align__(16) unsigned char wlds[];
    _Float16 *xh = reinterpret_cast<_Float16 *>(wlds);
    _Float16 *xl = xh + BM * kXS;
    _Float16 *xm = xl + BM * kXS;  // [BM][kXM]
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kq = lane >> 4, ln = lane & 15;
    const int n0 = blockIdx.x * (NW * 16 * WT) + w * 16 * WT;
    const int m0 = blockIdx.y * BM;
    const int nsteps = a.w.K / kStep, ks = gridDim.z;
    const int kb0 = int(blockIdx.z) * nsteps / ks, kb1 = (int(blockIdx.z) + 1) * nsteps / ks;

    XStage<BM, NTH, W::SPLIT> xs;
    xs.init(a.x, a.ldx, m0, a.M, t);
    f4_t acc[WT][MT];
#pragma unroll
    for (int j = 0; j < WT; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[j][mt] = f4_t{0.f, 0.f, 0.f, 0.f};

    typename W::Regs cur[WT], nxt[WT];
#pragma unroll
    for (int j = 0; j < WT; ++j) load_w<T, TL>(a.w, (n0 >> 4) + j, ln, kb0, kq, cur[j]);
    xs.load(kb0);
    if constexpr (W::MIN) xs.clear_sums(xm, t);
    for (int kb = kb0; kb < kb1; ++kb) {
        if (kb != kb0) lds_barrier();  // the previous step's reads of xh / xl / xm are done
        xs.template store<W::MIN>(xh, xl, xm);
        lds_barrier();
        // the next step's operands (past the end: the last step's again, never used, so that
        // no load sits behind a branch)
        const int kn = min(kb + 1, kb1 - 1);
#pragma unroll
        for (int j = 0; j < WT; ++j) load_w<T, TL>(a.w, (n0 >> 4) + j, ln, kn, kq, nxt[j]);
        xs.load(kn);
        block_mfma<T, MT, WT>(cur, xh, xl, xm, ln, kq, acc);
#pragma unroll
        for (int j = 0; j < WT; ++j) cur[j] = nxt[j];
    }
    if constexpr (MODE == 1) {
        // lane (kq, ln) holds rows mt 16 + 4 kq + r of columns n0 + 16 j + ln: its best over
        // its WT columns, then over the 16 lanes of the row group (DPP), then over the
        // waves (LDS; every wave's reads of the staged X are done first)
        float best[MT][4];
        uint32_t bidx[MT][4];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                best[mt][r] = -INFINITY;
                bidx[mt][r] = 0xffffffffu;
            }
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            const int n = n0 + 16 * j + ln;
            if (n >= a.w.N || n == a.mask_id) continue;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r) argmax_merge(best[mt][r], bidx[mt][r], acc[j][mt][r], uint32_t(n));
        }
        __syncthreads();
        float *mv = reinterpret_cast<float *>(wlds);                     // [waves][BM]
        uint32_t *mi = reinterpret_cast<uint32_t *>(mv + NW * BM);  // [waves][BM]
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = best[mt][r];
                uint32_t i = bidx[mt][r];
                argmax_merge(v, i, dpp_mov<kDppXor1>(v), dpp_mov<kDppXor1>(i));
                argmax_merge(v, i, dpp_mov<kDppXor2>(v), dpp_mov<kDppXor2>(i));
                argmax_merge(v, i, dpp_mov<kDppHalfMirror>(v), dpp_mov<kDppHalfMirror>(i));
                argmax_merge(v, i, dpp_mov<kDppMirror>(v), dpp_mov<kDppMirror>(i));
                if (ln == 0) {
                    mv[w * BM + mt * 16 + 4 * kq + r] = v;
                    mi[w * BM + mt * 16 + 4 * kq + r] = i;
                }
            }
        __syncthreads();
        if (t < BM && m0 + t < a.M) {  // ties -> the lowest index, so the merge order is free
            float v = mv[t];
            uint32_t i = mi[t];
#pragma unroll
            for (int w2 = 1; w2 < NW; ++w2) argmax_merge(v, i, mv[w2 * BM + t], mi[w2 * BM + t]);
            a.pv[size_t(m0 + t) * a.parts + blockIdx.x] = v;
            a.pi[size_t(m0 + t) * a.parts + blockIdx.x] = i;
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < WT; ++j) {
        const int n = n0 + 16 * j + ln;
        if (n >= a.w.N) continue;
        if (a.part) {
            float *pp = a.part + size_t(blockIdx.z) * a.M * a.w.N;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + mt * 16 + 4 * kq + r;
                    if (m < a.M) pp[size_t(m) * a.w.N + n] = acc[j][mt][r];
                }
            continue;
        }
        const float bv = a.bias ? a.bias[n] : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + mt * 16 + 4 * kq + r;
                if (m >= a.M) continue;
                float v = acc[j][mt][r] + bv;
                if (a.R) v += a.R[size_t(m) * a.ldr + n];
                if (a.relu) v = fmaxf(v, 0.f);
                a.y[size_t(m) * a.ldy + n] = v;
            }
    }
}

struct Tile {
    int bm, nw, wt;
    int cols() const { return 16 * nw * wt; }
    int blocks(int N, int M) const { return (N + cols() - 1) / cols() * ((M + bm - 1) / bm); }
};
// The tile for a product: 256 columns of W per workgroup, so that X is staged least often,
// where at least 96 such tiles, or those times the K steps that can be split off (split_k),
// keep the device busy, else 64 columns.  Measured (us, 256 / 64 columns): q4_K 8192 x 2048 at
// 1651 rows 159 / 192, q6_K 1024 x 4096 at 911 rows 38.8 / 43.6; below the line q4_K 1024 x 1024
// at 911 rows 17.1 / 15.9.  (Just 256 pieces in 16 splits: q6_K 1024 x 4096 at 203 rows 18.2,
// in 8 of 64 columns 15.9; in 8 or 32 splits the wide tiles are as good or better.)  A product
// is split only where it has fewer than 256 tiles of 64
// columns, or 96 to 128 of 256 (two halves then beat both the unsplit wide tiles and, from K =
// 2048, the narrow ones: q4_K 2048 x 2048 at 832 rows 29.0 / 38.2 / 31.7 us): the context's
// workspace holds one product's planes at a time, and the others stay independent of it
// (q4_K 4096 x 1024 at 203 rows: 13.7 split / 14.2).
Tile tile_of(const DevMatrix &w, int M) {
    if (M <= 16) return {16, 4, 1};
    if (M <= 32) return {32, 4, 1};
    const Tile wide{64, 8, 2}, narrow{64, 4, 1};
    const int nw = wide.blocks(w.N, M);
    const int64_t pieces = int64_t(nw) * (w.K / kStep);
    const bool split = narrow.blocks(w.N, M) < 256 && (pieces > 256 || (pieces == 256 && nw != 16));
    return nw >= 96 || split ? wide : narrow;
}

template <int T, int BM, int NW, int WT, bool TL, int MODE = 0>
hipError_t launch_t(const MfmaArgs &a, int ks, hipStream_t st) {
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mfma<T, BM, NW, WT, TL, MODE>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(mfma_lds<BM>()));
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((k_mfma<T, BM, NW, WT, TL, MODE>),
                       dim3((a.w.N + 16 * NW * WT - 1) / (16 * NW * WT), (a.M + BM - 1) / BM, ks), dim3(NW * 64),
                       mfma_lds<BM>(), st, a);
    return hipGetLastError();
}

template <int T, bool TL>
hipError_t launch_tl(const MfmaArgs &a, const Tile &t, int ks, hipStream_t st) {
    if (t.bm == 16) return launch_t<T, 16, 4, 1, TL>(a, ks, st);
    if (t.bm == 32) return launch_t<T, 32, 4, 1, TL>(a, ks, st);
    return t.nw == 4 ? launch_t<T, 64, 4, 1, TL>(a, ks, st) : launch_t<T, 64, 8, 2, TL>(a, ks, st);
}

// q6_K / q4_K with its tile-major copy reads that copy
template <int T>
hipError_t launch(const MfmaArgs &a, const Tile &t, int ks, hipStream_t st) {
    if constexpr (T == GGML_Q6_K || T == GGML_Q4_K) {
        if (a.w.t) return launch_tl<T, true>(a, t, ks, st);
    }
    return launch_tl<T, false>(a, t, ks, st);
}

// Split-K reduction fused with the decoder's residual add and the next LayerNorm
// (src/model.rs:183-187): y = sum_z part[z][m] (in z order) + bias; x[m] += y;
// h[m] = LayerNorm(x[m]) with biased variance (f64 statistics).  One workgroup of 256
// threads per row, each thread on float4 slots t + 256 c; N <= 4096, N % 4 == 0.
__global__ __launch_bounds__(256) void k_splitk_residual_ln(const float *part, int ks, int M, int N,
                                                             const float *bias, float *x, const float *g,
                                                             const float *b, float eps, float *h) {
    __shared__ double red[8];
    const int m = blockIdx.x;
    const size_t mn = size_t(M) * N, off = size_t(m) * N;
    float4 *xr = reinterpret_cast<float4 *>(x + off);
    auto form = [&](int f) {
        // the partials requested eight at a time, then added in z order
        float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int z0 = 0; z0 < ks; z0 += 8) {
            float4 p8[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                p8[u] = z0 + u < ks ? ld4(part + size_t(z0 + u) * mn + off, f) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (z0 + u < ks) {
                    if (z0 + u == 0) y = p8[u];
                    else add4(y, p8[u]);
                }
        }
        if (bias) add4(y, ld4(bias, f));
        float4 v = xr[f];
        add4(v, y);
        return v;
    };
    workgroup_row_layernorm<4>(N, form, [&](int f, const float4 &v) { xr[f] = v; }, g, b, eps, h + off, red);
}

// Split-K reduction of the fused QKV projection written straight into q [M][d] and
// the caches at slot *step (kernels/malaga.cu:142-154): f16 (rounded to nearest even) or
// f32 (the generic path's caches).
__device__ __forceinline__ void store_kv(__half *p, float v) { *p = __float2half(v); }
__device__ __forceinline__ void store_kv(float *p, float v) { *p = v; }

template <typename KT>
__global__ __launch_bounds__(256) void k_splitk_qkv(const float *part, int ks, int M, int d, const float *bias, int H,
                                                     int hd, int slots, const uint32_t *step, float *q, KT *kc,
                                                     KT *vc) {
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x, N = size_t(3) * d, mn = size_t(M) * N;
    if (i >= mn) return;
    const int m = int(i / N), c = int(i % N);
    float v = 0.f;
    for (int z0 = 0; z0 < ks; z0 += 8) {
        float p8[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p8[u] = z0 + u < ks ? part[size_t(z0 + u) * mn + i] : 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (z0 + u < ks) v = (z0 + u == 0) ? p8[u] : v + p8[u];
    }
    if (bias) v += bias[c];
    if (c < d) {
        q[size_t(m) * d + c] = v;
    } else {
        const int cc = c < 2 * d ? c - d : c - 2 * d;
        const size_t o = ((size_t(m) * H + cc / hd) * slots + *step) * hd + cc % hd;
        store_kv((c < 2 * d ? kc : vc) + o, v);
    }
}

// K splits that fill the device, within the workspace.  The small tiles: at least one
// workgroup per CU.  The 64-row tiles: what 256 workgroups allow, but one or two steps of K
// per workgroup in the fewest splits that have no more: each adds a plane to write and read
// (q6_K 1024 x 1024 at 300 rows 11.1 us in 2 splits, 11.7 in 3, 11.3 in 4, 14.4 unsplit; 1024
// x 4096 at 300 rows, wide, 19.6 in 8 splits, 23.4 in 12).  A second workgroup of 4 waves on a
// CU only where chains of 3 or more steps are left (512 x 2048 at 832 rows: 17.1 us with 416
// workgroups of 2 steps, 21.3 with 208 of 4; but 1024 x 1024 at 512 rows: 13.4 with 512 of 1
// step, 12.3 with 256 of 2).
//
// reduced: the planes are added up by a kernel that runs in any case (launch_split).  Two
// halves then also where 129 to 255 tiles of 64 columns could do without (q4_K 1024 x 1024 at
// 911 rows with the residual and LayerNorm 18.2 us, 25.1 unsplit).
int split_k(const DevMatrix &w, int M, size_t ws_bytes, bool reduced = false) {
    const Tile t = tile_of(w, M);
    const int base = t.blocks(w.N, M), nsteps = w.K / kStep;
    auto ceil_div = [](int a, int b) { return (a + b - 1) / b; };
    int ks = 1;
    if (base < 256 && t.bm < 64) {
        ks = std::min(nsteps, ceil_div(256, base));
    } else if (base < 256) {
        ks = std::min(nsteps, 256 / base);
        int s = ceil_div(nsteps, ks);
        if (t.nw == 4 && s >= 3 && ks > 1) {
            ks = std::min(nsteps, 512 / base);
            s = std::max(2, ceil_div(nsteps, ks));
        }
        if (s <= 2) ks = ceil_div(nsteps, s);
        if (reduced && ks == 1 && t.nw == 4) ks = std::min(nsteps, 2);
    }
    while (ks > 1 && size_t(ks) * M * w.N * sizeof(float) > ws_bytes) --ks;
    return ks;
}

// ---------------------------------------------------------------- resident X
//
// Decode batches (M <= 32) with K small enough that all of X fits in LDS as hi/lo
// f16 (BM * K * 4 bytes <= ~140 KB): one persistent workgroup of 8 waves per CU
// stages X once, then every wave streams 16-row tiles of W (tile t, t + waves, ...)
// with the next (tile, K-step) in flight in registers.  No split K, no reduction
// kernel, and X is read from HBM/L2 once per workgroup instead of once per tile.
// MODE 0 stores Y (bias, residual, ReLU); MODE 1 keeps a running argmax per X row
// (the greedy LM head) and writes one partial per workgroup (its waves' merged in LDS).

constexpr int kRxWaves = 8;
constexpr int kRxDepth = 2;  // (group, K-step) jobs of W in flight per wave
// 16-row tiles of W per job (reuse of each X fragment), sized to the registers a
// type's raw K step needs; q6_K issues 14 loads per tile and K step, and a wave
// tracks at most 63 outstanding loads (kRxDepth x tiles x loads must stay below,
// or every job waits for all loads in flight)
template <int T>
constexpr int rx_nt() { return T == GGML_F16 ? 1 : (T == GGML_Q8_0 || T == GGML_Q6_K) ? 2 : 4; }
constexpr size_t kRxMaxLds = 150 * 1024;

struct RxArgs {
    WPtr w;
    const float *x;
    int ldx, M;
    float *y;
    int ldy;
    const float *bias, *R;
    int ldr, relu;
    int mask_id;      // MODE 1: row index never selected (-1: none)
    float *pv;        // MODE 1: partials [M][parts]
    uint32_t *pi;
    int parts;
    bool nt;          // MODE 1: the weights do not stay in the cache until the next step
};

// halves per staged X row: 8 mod 64 dwords, where the A reads (16 rows x 4 k-groups of
// 16 bytes) meet no bank conflict (K + 8: 5.4 M conflict cycles per LM-head launch)
__host__ __device__ constexpr int rx_stride(int K) { return K + 16; }

size_t rx_lds_bytes(int BM, int K) {
    return size_t(BM) * rx_stride(K) * 2 * sizeof(_Float16) + size_t(K / 16) * BM * sizeof(float);
}

template <int T, int BM, int MODE, bool TL, bool NT>
__global__ __launch_bounds__(kRxWaves * 64) void k_mfma_rx(RxArgs a) {
    using W = MW<T>;
    constexpr int MT = BM / 16;
    constexpr int kRxNT = rx_nt<T>();
    extern __shared__ __align__(16) unsigned char rx_lds[];
    const int K = a.w.K, XS = rx_stride(K);
    _Float16 *xh = reinterpret_cast<_Float16 *>(rx_lds);
    _Float16 *xl = xh + BM * XS;
    float *xsum = reinterpret_cast<float *>(xl + BM * XS);  // [K / 16][BM]
    const int t = threadIdx.x, lane = t & 63;
    const int kq = lane >> 4, ln = lane & 15;
    const int nsteps = K / kStep;
    const int ngroups = (a.w.N + 16 * kRxNT - 1) / (16 * kRxNT);  // groups of kRxNT 16-row tiles
    // a scalar: the job loop's bounds stay uniform (no divergent load paths)
    const int gw = __builtin_amdgcn_readfirstlane(blockIdx.x * kRxWaves + (t >> 6)), nw = gridDim.x * kRxWaves;
    const int njobs = gw < ngroups ? ((ngroups - 1 - gw) / nw + 1) * nsteps : 0;  // (group, step) pairs of this wave

    typename W::Regs ring[kRxDepth][kRxNT];
    auto job_base = [&](int j) { return (gw + (j / nsteps) * nw) * 16 * kRxNT; };
    auto load_job = [&](int j, typename W::Regs (&r)[kRxNT]) {
#pragma unroll
        for (int nt = 0; nt < kRxNT; ++nt) load_w<T, TL, NT>(a.w, (job_base(j) >> 4) + nt, ln, j % nsteps, kq, r[nt]);
    };

    // stage X: chunks of 8 values, one 16-byte store each (consecutive lanes: consecutive
    // chunks of a row, so a store of 16 lanes covers 256 contiguous bytes of LDS: no bank
    // conflicts), up to 4 per thread in flight.  Chunk c of a row holds x[8 c .. 8 c + 7], or
    // for split-B types the two 4-value groups split_pos puts there.  BM K / 8 is a multiple
    // of the 512 threads, so every lane runs the same trips (the DPP sums below need them all).
    {
        const int cpr = K / 8, nch = BM * cpr;
        auto koff = [](int c, int half) {
            if constexpr (W::SPLIT) return 32 * (c >> 2) + 16 * half + 4 * (c & 3);
            else return 8 * c + 4 * half;
        };
        for (int c0 = t; c0 < nch; c0 += kRxWaves * 64 * 4) {
            float4 v[4][2];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = c0 + u * kRxWaves * 64;
                const int m = c / cpr, cc = c % cpr;
                const bool ok = c < nch && m < a.M;
                const float *src = a.x + size_t(ok ? m : 0) * a.ldx;
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    v[u][f] = ok ? *reinterpret_cast<const float4 *>(src + koff(cc, f)) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = c0 + u * kRxWaves * 64;
                if (c >= nch) break;  // the same trips in every lane
                const int m = c / cpr, cc = c % cpr;
                const float e[8] = {v[u][0].x, v[u][0].y, v[u][0].z, v[u][0].w,
                                    v[u][1].x, v[u][1].y, v[u][1].z, v[u][1].w};
                h8_t hv, lv;
                split_h8(e, hv, lv);
                *reinterpret_cast<h8_t *>(xh + m * XS + 8 * cc) = hv;
                *reinterpret_cast<h8_t *>(xl + m * XS + 8 * cc) = lv;
                if constexpr (W::MIN) {  // 16-value sums: this chunk and the next (lane t ^ 1)
                    float sm = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
                    sm += dpp_mov<kDppXor1>(sm);
                    if (!(cc & 1)) xsum[(cc >> 1) * BM + m] = sm;
                }
            }
        }
    }
    __syncthreads();
    // the first kRxDepth (group, K-step) jobs of W: requested once X is staged, so that
    // the job loop is entered with the same loads in flight as on every later trip
    // (requested before the staging, they made the compiler wait for every load at the
    // top of each job: 2 of the ring's jobs in flight became 0)
    // (unconditional: a job past this wave's last reads a clamped row and is never used;
    // a skipped request would leave the compiler unsure how many loads follow each one)
#pragma unroll
    for (int u = 0; u < kRxDepth; ++u) {
        load_job(u, ring[u]);
        __builtin_amdgcn_sched_barrier(0);  // jobs requested in order
    }

    f4_t acc[MT][kRxNT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < kRxNT; ++nt) acc[mt][nt] = f4_t{0.f, 0.f, 0.f, 0.f};
    float best[MT][4];
    uint32_t bidx[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            best[mt][r] = -INFINITY;
            bidx[mt][r] = 0xffffffffu;
        }

    // job j uses ring slot j % kRxDepth, refilled with job j + kRxDepth once consumed;
    // each X fragment read from LDS feeds kRxNT tiles of W
    auto job = [&](int j, const typename W::Regs (&cur)[kRxNT]) {
        const int kb = j % nsteps;
        if constexpr (W::SPLIT) {
            // the block's 8 split-B slices chain in the MFMA's C operand; d once per block
            f4_t cb[MT][kRxNT];
            // A fragments of slice s + 1 are read from LDS while slice s runs on the MFMA
            h8_t ahs[2][MT], als[2][MT];
            auto read_a = [&](int s, h8_t (&ah)[MT], h8_t (&al)[MT]) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const int xo = (mt * 16 + ln) * XS + kb * kStep + 32 * s + 8 * kq;
                    ah[mt] = *reinterpret_cast<const h8_t *>(xh + xo);
                    al[mt] = *reinterpret_cast<const h8_t *>(xl + xo);
                }
            };
            read_a(0, ahs[0], als[0]);
#pragma unroll
            for (int s = 0; s < W::SLICES32; ++s) {
                if (s + 1 < W::SLICES32) read_a(s + 1, ahs[(s + 1) & 1], als[(s + 1) & 1]);
                h8_t bh[kRxNT], bl[kRxNT];
#pragma unroll
                for (int nt = 0; nt < kRxNT; ++nt) W::b_split(cur[nt], s, bh[nt], bl[nt]);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const h8_t ah = ahs[s & 1][mt], al = als[s & 1][mt];
#pragma unroll
                    for (int nt = 0; nt < kRxNT; ++nt)
                        cb[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            ah, bh[nt], s ? cb[mt][nt] : f4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (int nt = 0; nt < kRxNT; ++nt)
                        cb[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh[nt], cb[mt][nt], 0, 0, 0);
#pragma unroll
                    for (int nt = 0; nt < kRxNT; ++nt)
                        cb[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl[nt], cb[mt][nt], 0, 0, 0);
                }
            }
#pragma unroll
            for (int nt = 0; nt < kRxNT; ++nt) {
                const float d = W::d_of(cur[nt]);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[mt][nt][r] = fmaf(d, cb[mt][nt][r], acc[mt][nt][r]);
            }
        } else {
#pragma unroll
            for (int s = 0; s < W::SLICES; ++s) {
                float sc[kRxNT], mn[kRxNT];
                decltype(W::b(cur[0], s)) bop[kRxNT];
#pragma unroll
                for (int nt = 0; nt < kRxNT; ++nt) {
                    W::scale(cur[nt], s, sc[nt], mn[nt]);
                    bop[nt] = W::b(cur[nt], s);
                }
                const int kx = kb * kStep + s * W::SK;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const int xo = (mt * 16 + ln) * XS + kx + kq * (W::SK / 4);
                    const float *xsp = xsum + (kx >> 4) * BM + mt * 16 + 4 * kq;
                    float4 xsv = make_float4(0.f, 0.f, 0.f, 0.f);
                    if constexpr (W::MIN) {
                        xsv = *reinterpret_cast<const float4 *>(xsp);
                        if constexpr (W::SK == 32) {
                            const float4 x2 = *reinterpret_cast<const float4 *>(xsp + BM);
                            xsv = make_float4(xsv.x + x2.x, xsv.y + x2.y, xsv.z + x2.z, xsv.w + x2.w);
                        }
                    }
                    if constexpr (W::SK == 32) {
                        const h8_t ah = *reinterpret_cast<const h8_t *>(xh + xo), al = *reinterpret_cast<const h8_t *>(xl + xo);
#pragma unroll
                        for (int nt = 0; nt < kRxNT; ++nt) {
                            f4_t tmp = f4_t{0.f, 0.f, 0.f, 0.f};
                            tmp = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bop[nt], tmp, 0, 0, 0);
                            tmp = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bop[nt], tmp, 0, 0, 0);
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                acc[mt][nt][r] = W::MIN ? fmaf(sc[nt], tmp[r], fmaf(-mn[nt], (&xsv.x)[r], acc[mt][nt][r]))
                                                        : fmaf(sc[nt], tmp[r], acc[mt][nt][r]);
                        }
                    } else {
                        const h4_t ah = *reinterpret_cast<const h4_t *>(xh + xo), al = *reinterpret_cast<const h4_t *>(xl + xo);
#pragma unroll
                        for (int nt = 0; nt < kRxNT; ++nt) {
                            f4_t tmp = f4_t{0.f, 0.f, 0.f, 0.f};
                            tmp = __builtin_amdgcn_mfma_f32_16x16x16f16(ah, bop[nt], tmp, 0, 0, 0);
                            tmp = __builtin_amdgcn_mfma_f32_16x16x16f16(al, bop[nt], tmp, 0, 0, 0);
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                acc[mt][nt][r] = W::MIN ? fmaf(sc[nt], tmp[r], fmaf(-mn[nt], (&xsv.x)[r], acc[mt][nt][r]))
                                                        : fmaf(sc[nt], tmp[r], acc[mt][nt][r]);
                        }
                    }
                }
            }
        }
        if (kb == nsteps - 1) {  // group done
#pragma unroll
            for (int nt = 0; nt < kRxNT; ++nt) {
                const int n = job_base(j) + nt * 16 + ln;
                if (n < a.w.N) {
                    // MODE 1 (the tied LM head) has no bias: no global load in this
                    // epilogue, which would make every later job wait for all loads
                    float bv = 0.f;
                    if constexpr (MODE == 0) bv = a.bias ? a.bias[n] : 0.f;
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int m = mt * 16 + 4 * kq + r;
                            float v = acc[mt][nt][r] + bv;
                            if constexpr (MODE == 0) {
                                if (m < a.M) {
                                    if (a.R) v += a.R[size_t(m) * a.ldr + n];
                                    if (a.relu) v = fmaxf(v, 0.f);
                                    a.y[size_t(m) * a.ldy + n] = v;
                                }
                            } else {
                                if (n != a.mask_id) argmax_merge(best[mt][r], bidx[mt][r], v, uint32_t(n));
                            }
                        }
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = f4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
    };
    // Main loop: every job is followed by its slot's refill.  The last jobs run in a
    // separate tail, so that no job in the main loop follows a skipped refill: the
    // compiler would then merge the two load states and wait for every load in
    // flight (the refills included) at the top of each job.
    int j0 = 0;
    for (; j0 + 2 * kRxDepth <= njobs; j0 += kRxDepth) {
#pragma unroll
        for (int u = 0; u < kRxDepth; ++u) {
            job(j0 + u, ring[u]);
            __builtin_amdgcn_sched_barrier(0);
            load_job(j0 + u + kRxDepth, ring[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; j0 < njobs; j0 += kRxDepth) {
#pragma unroll
        for (int u = 0; u < kRxDepth; ++u) {
            const int j = j0 + u;
            if (j >= njobs) break;  // wave-uniform
            job(j, ring[u]);
            if (j + kRxDepth < njobs) load_job(j + kRxDepth, ring[u]);
        }
    }
    if constexpr (MODE == 1) {
        // lanes 16 kq .. 16 kq + 15 hold the same X rows: reduce within each 16-lane row,
        // then over the workgroup's waves (LDS; the staged X is no longer read), so the
        // finalize merges one partial per workgroup and row
        __syncthreads();  // every wave's last reads of the staged X are done
        float *mv = reinterpret_cast<float *>(rx_lds);                  // [kRxWaves][BM]
        uint32_t *mi = reinterpret_cast<uint32_t *>(mv + kRxWaves * BM);  // [kRxWaves][BM]
        const int wv = t >> 6;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = best[mt][r];
                uint32_t i = bidx[mt][r];
                argmax_merge(v, i, dpp_mov<kDppXor1>(v), dpp_mov<kDppXor1>(i));
                argmax_merge(v, i, dpp_mov<kDppXor2>(v), dpp_mov<kDppXor2>(i));
                argmax_merge(v, i, dpp_mov<kDppHalfMirror>(v), dpp_mov<kDppHalfMirror>(i));
                argmax_merge(v, i, dpp_mov<kDppMirror>(v), dpp_mov<kDppMirror>(i));
                const int m = mt * 16 + 4 * kq + r;
                if (ln == 0) {
                    mv[wv * BM + m] = v;
                    mi[wv * BM + m] = i;
                }
            }
        __syncthreads();
        if (t < BM && t < a.M) {  // ties -> the lowest index, so the order of the merge is free
            float v = mv[t];
            uint32_t i = mi[t];
#pragma unroll
            for (int w2 = 1; w2 < kRxWaves; ++w2) argmax_merge(v, i, mv[w2 * BM + t], mi[w2 * BM + t]);
            a.pv[size_t(t) * a.parts + blockIdx.x] = v;
            a.pi[size_t(t) * a.parts + blockIdx.x] = i;
        }
    }
}

// Dynamic LDS beyond 64 KB needs the kernel attribute raised once.
template <int T, int BM, int MODE, bool TL, bool NT>
hipError_t launch_rx_bm(const RxArgs &a, int grid, hipStream_t st) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mfma_rx<T, BM, MODE, TL, NT>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(kRxMaxLds));
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((k_mfma_rx<T, BM, MODE, TL, NT>), dim3(grid), dim3(kRxWaves * 64), rx_lds_bytes(BM, a.w.K), st,
                       a);
    return hipGetLastError();
}

template <int T, int MODE, bool TL, bool NT = false>
hipError_t launch_rx_tl(const RxArgs &a, int M, int grid, hipStream_t st) {
    return M <= 16 ? launch_rx_bm<T, 16, MODE, TL, NT>(a, grid, st) : launch_rx_bm<T, 32, MODE, TL, NT>(a, grid, st);
}

template <int T, int MODE>
hipError_t launch_rx(const RxArgs &a, int M, int grid, hipStream_t st) {
    if constexpr (T == GGML_Q6_K || T == GGML_Q4_K) {
        if constexpr (T == GGML_Q6_K && MODE == 1)
            if (a.w.t && a.nt) return launch_rx_tl<T, MODE, true, true>(a, M, grid, st);
        if (a.w.t) return launch_rx_tl<T, MODE, true>(a, M, grid, st);
    }
    return launch_rx_tl<T, MODE, false>(a, M, grid, st);
}

int rx_nt_of(uint32_t t) {
    switch (t) {
    case GGML_F16: return rx_nt<GGML_F16>();
    case GGML_Q8_0: return rx_nt<GGML_Q8_0>();
    case GGML_Q6_K: return rx_nt<GGML_Q6_K>();
    case GGML_Q5_K: return rx_nt<GGML_Q5_K>();
    default: return rx_nt<GGML_Q4_K>();
    }
}

int rx_grid(const DevMatrix &w, int M) {
    const int bm = M <= 16 ? 16 : 32;
    const size_t lds = rx_lds_bytes(bm, w.K);
    const int per_cu = lds * 2 <= 160 * 1024 ? 2 : 1;
    const int nt = rx_nt_of(w.type);
    const int groups = (w.N + 16 * nt - 1) / (16 * nt);
    const int waves = std::min(groups, 256 * per_cu * kRxWaves);
    return (waves + kRxWaves - 1) / kRxWaves;
}

}  // namespace

bool gemm_mfma_supported(const DevMatrix &w) {
    const bool type_ok = w.type == GGML_Q4_K || w.type == GGML_Q5_K || w.type == GGML_Q6_K ||
                         w.type == GGML_Q8_0 || w.type == GGML_F16;
    return type_ok && w.K % kStep == 0 && w.N > 0;
}

bool gemm_rx_supported(const DevMatrix &w, int M) {
    return gemm_mfma_supported(w) && M >= 1 && M <= 32 && rx_lds_bytes(M <= 16 ? 16 : 32, w.K) <= kRxMaxLds;
}

// Stored products take the resident-X kernel only when W is large enough to keep
// every CU busy (staging X per workgroup is then amortised); smaller matrices use
// the split-K tile kernel.
constexpr int kRxMinRows = 65536;

namespace {
template <int MODE>
hipError_t run_rx(const DevMatrix &w, RxArgs &a, int M, int grid, hipStream_t st) {
    switch (w.type) {
    case GGML_Q4_K: return launch_rx<GGML_Q4_K, MODE>(a, M, grid, st);
    case GGML_Q5_K: return launch_rx<GGML_Q5_K, MODE>(a, M, grid, st);
    case GGML_Q6_K: return launch_rx<GGML_Q6_K, MODE>(a, M, grid, st);
    case GGML_Q8_0: return launch_rx<GGML_Q8_0, MODE>(a, M, grid, st);
    case GGML_F16: return launch_rx<GGML_F16, MODE>(a, M, grid, st);
    default: return hipErrorInvalidValue;
    }
}
RxArgs rx_args(const DevMatrix &w, const float *X, int ldx, int M) {
    RxArgs a{};
    a.w = wptr_of(w);
    a.x = X;
    a.ldx = ldx;
    a.M = M;
    a.mask_id = -1;
    return a;
}
}  // namespace

// 33..64 rows: the wide-tile kernel with the argmax epilogue (X staged per K step)
namespace {
constexpr int kWArgmaxMaxRows = 64;
bool w_argmax_rows(const DevMatrix &w, int M) {
    return !gemm_rx_supported(w, M) && gemm_mfma_supported(w) && M > 32 && M <= kWArgmaxMaxRows;
}
constexpr Tile kWArgmaxTile{64, 8, 2};  // X is staged least often
int w_argmax_grid(const DevMatrix &w) { return kWArgmaxTile.blocks(w.N, 1); }

template <int T>
hipError_t launch_w_argmax(const MfmaArgs &a, int M, hipStream_t st) {
    if constexpr (T == GGML_Q6_K || T == GGML_Q4_K) {
        if (a.w.t) return launch_t<T, 64, 8, 2, true, 1>(a, 1, st);
    }
    return launch_t<T, 64, 8, 2, false, 1>(a, 1, st);
}
}  // namespace

bool gemm_argmax_supported(const DevMatrix &w, int M) { return gemm_rx_supported(w, M) || w_argmax_rows(w, M); }

// one partial per workgroup
int gemm_argmax_parts(const DevMatrix &w, int M) { return w_argmax_rows(w, M) ? w_argmax_grid(w) : rx_grid(w, M); }

hipError_t gemm_argmax(const DevMatrix &w, const float *X, int ldx, int M, int mask_id, float *pv, uint32_t *pi,
                       int *parts, hipStream_t st) {
    if (!gemm_argmax_supported(w, M) || ldx % 4 || reinterpret_cast<uintptr_t>(X) % 16) return hipErrorInvalidValue;
    if (w_argmax_rows(w, M)) {
        MfmaArgs a{};
        a.w = wptr_of(w);
        a.x = X;
        a.ldx = ldx;
        a.M = M;
        a.mask_id = mask_id;
        a.pv = pv;
        a.pi = pi;
        a.parts = w_argmax_grid(w);
        *parts = a.parts;
        switch (w.type) {
        case GGML_Q4_K: return launch_w_argmax<GGML_Q4_K>(a, M, st);
        case GGML_Q5_K: return launch_w_argmax<GGML_Q5_K>(a, M, st);
        case GGML_Q6_K: return launch_w_argmax<GGML_Q6_K>(a, M, st);
        case GGML_Q8_0: return launch_w_argmax<GGML_Q8_0>(a, M, st);
        case GGML_F16: return launch_w_argmax<GGML_F16>(a, M, st);
        default: return hipErrorInvalidValue;
        }
    }
    // A step reads the decoder layers and the head, and what of both exceeds the Infinity Cache
    // is read from memory again: with ordinary loads the head evicts the layers.  Read
    // non-temporally it leaves them there, and costs its own share of the cache.  32 sentences,
    // 32 tokens, ordinary / non-temporal (d = 1024): 12 layers and 221 MB of head (333 MB) 19.05 /
    // 18.15 ms, 197 MB in all 17.5 / 17.4 (8 sentences 15.3 / 14.8); but 2 layers and 192 MB 5.09 /
    // 5.42, 151 MB 6.82 / 7.11: so from three quarters of the 256 MB.  (A head by itself, over and
    // over, is faster with what the cache keeps.)
    constexpr size_t kCacheKeeps = 192'000'000;
    RxArgs a = rx_args(w, X, ldx, M);
    a.nt = w.beside > 0 && tile_major_bytes(w.type, w.N, w.K) + w.beside > kCacheKeeps;
    a.mask_id = mask_id;
    a.pv = pv;
    a.pi = pi;
    const int grid = rx_grid(w, M);
    a.parts = grid;
    *parts = a.parts;
    return run_rx<1>(w, a, M, grid, st);
}

hipError_t gemm_mfma(const DevMatrix &w, const float *X, int ldx, int M, float *Y, int ldy, const float *bias,
                     bool relu, const float *R, int ldr, hipStream_t st, float *ws, size_t ws_bytes) {
    if (M <= 0) return hipSuccess;
    if (!gemm_mfma_supported(w) || ldx % 4 || reinterpret_cast<uintptr_t>(X) % 16) return hipErrorInvalidValue;
    if (gemm_rx_supported(w, M) && w.N >= kRxMinRows) {
        RxArgs r = rx_args(w, X, ldx, M);
        r.y = Y;
        r.ldy = ldy;
        r.bias = bias;
        r.R = R;
        r.ldr = ldr;
        r.relu = relu ? 1 : 0;
        return run_rx<0>(w, r, M, rx_grid(w, M), st);
    }
    MfmaArgs a{};
    a.w = wptr_of(w);
    a.x = X;
    a.ldx = ldx;
    a.M = M;
    a.y = Y;
    a.ldy = ldy;
    a.bias = bias;
    a.R = R;
    a.ldr = ldr;
    a.relu = relu ? 1 : 0;
    const int ks = ws ? split_k(w, M, ws_bytes) : 1;
    a.part = ks > 1 ? ws : nullptr;
    hipError_t e;
    switch (w.type) {
    case GGML_Q4_K: e = launch<GGML_Q4_K>(a, tile_of(w, M), ks, st); break;
    case GGML_Q5_K: e = launch<GGML_Q5_K>(a, tile_of(w, M), ks, st); break;
    case GGML_Q6_K: e = launch<GGML_Q6_K>(a, tile_of(w, M), ks, st); break;
    case GGML_Q8_0: e = launch<GGML_Q8_0>(a, tile_of(w, M), ks, st); break;
    case GGML_F16: e = launch<GGML_F16>(a, tile_of(w, M), ks, st); break;
    default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess || ks == 1) return e;
    const size_t mn = size_t(M) * w.N;
    hipLaunchKernelGGL(k_splitk_reduce, dim3(unsigned((mn + 255) / 256)), dim3(256), 0, st, ws, ks, M, w.N, bias, R,
                       ldr, relu ? 1 : 0, Y, ldy);
    return hipGetLastError();
}


namespace {
// Runs the tile kernel with K split over workgroups into ws; returns the split
// count (1: not split, nothing launched).
int launch_split(const DevMatrix &w, const float *X, int ldx, int M, hipStream_t st, float *ws, size_t ws_bytes,
                 hipError_t *err) {
    *err = hipSuccess;
    if (!ws || !gemm_mfma_supported(w) || ldx % 4 || reinterpret_cast<uintptr_t>(X) % 16) return 1;
    if (gemm_rx_supported(w, M) && w.N >= kRxMinRows) return 1;
    const int ks = split_k(w, M, ws_bytes, true);
    if (ks <= 1) return 1;
    MfmaArgs a{};
    a.w = wptr_of(w);
    a.x = X;
    a.ldx = ldx;
    a.M = M;
    a.part = ws;
    switch (w.type) {
    case GGML_Q4_K: *err = launch<GGML_Q4_K>(a, tile_of(w, M), ks, st); break;
    case GGML_Q5_K: *err = launch<GGML_Q5_K>(a, tile_of(w, M), ks, st); break;
    case GGML_Q6_K: *err = launch<GGML_Q6_K>(a, tile_of(w, M), ks, st); break;
    case GGML_Q8_0: *err = launch<GGML_Q8_0>(a, tile_of(w, M), ks, st); break;
    case GGML_F16: *err = launch<GGML_F16>(a, tile_of(w, M), ks, st); break;
    default: return 1;
    }
    return ks;
}
}  // namespace

hipError_t gemm_residual_ln(const DevMatrix &w, const float *X, int ldx, int M, const float *bias, float *x,
                            const float *g, const float *b, float eps, float *h, hipStream_t st, float *ws,
                            size_t ws_bytes) {
    if (M <= 0) return hipSuccess;
    if (w.N > 4096 || w.N % 4) return hipErrorInvalidValue;
    hipError_t e;
    const int ks = launch_split(w, X, ldx, M, st, ws, ws_bytes, &e);
    if (e != hipSuccess) return e;
    if (ks > 1) {
        hipLaunchKernelGGL(k_splitk_residual_ln, dim3(M), dim3(256), 0, st, ws, ks, M, w.N, bias, x, g, b, eps, h);
        return hipGetLastError();
    }
    // x = x + X W^T + bias in place (R = Y = x), then the LayerNorm
    e = gemm(w, X, ldx, M, x, w.N, bias, false, x, w.N, st, ws, ws_bytes);
    if (e != hipSuccess) return e;
    return layernorm(x, M, w.N, g, b, eps, h, st);
}

namespace {
template <typename KT>
hipError_t gemm_qkv_t(const DevMatrix &w, const float *X, int ldx, int M, const float *bias, int H, int hd, int slots,
                      const uint32_t *step, float *q, KT *kc, KT *vc, float *qkv_tmp, hipStream_t st, float *ws,
                      size_t ws_bytes) {
    if (M <= 0) return hipSuccess;
    const int d = H * hd;
    if (w.N != 3 * d) return hipErrorInvalidValue;
    hipError_t e;
    const int ks = launch_split(w, X, ldx, M, st, ws, ws_bytes, &e);
    if (e != hipSuccess) return e;
    if (ks > 1) {
        const size_t n = size_t(M) * w.N;
        hipLaunchKernelGGL(k_splitk_qkv<KT>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, ws, ks, M, d, bias, H,
                           hd, slots, step, q, kc, vc);
        return hipGetLastError();
    }
    e = gemm(w, X, ldx, M, qkv_tmp, w.N, bias, false, nullptr, 0, st, ws, ws_bytes);
    if (e != hipSuccess) return e;
    return qkv_split(qkv_tmp, M, H, hd, slots, step, q, kc, vc, st);
}
}  // namespace

hipError_t gemm_qkv(const DevMatrix &w, const float *X, int ldx, int M, const float *bias, int H, int hd, int slots,
                    const uint32_t *step, float *q, __half *kc, __half *vc, float *qkv_tmp, hipStream_t st, float *ws,
                    size_t ws_bytes) {
    return gemm_qkv_t(w, X, ldx, M, bias, H, hd, slots, step, q, kc, vc, qkv_tmp, st, ws, ws_bytes);
}

hipError_t gemm_qkv(const DevMatrix &w, const float *X, int ldx, int M, const float *bias, int H, int hd, int slots,
                    const uint32_t *step, float *q, float *kc, float *vc, float *qkv_tmp, hipStream_t st, float *ws,
                    size_t ws_bytes) {
    return gemm_qkv_t(w, X, ldx, M, bias, H, hd, slots, step, q, kc, vc, qkv_tmp, st, ws, ws_bytes);
}

}  // namespace mlg
