// Chunked (WY / UT) Gated DeltaNet prefill on the matrix cores.
//
// The reference runs prefill as a token-serial scan (gdn_scan_batch2,
// LLM/metal/Kernels.metal:1570-1625; GDN.step, LLM/src/SIMD/GDN.swift:71-109).
// Unrolling that recurrence over a chunk of L tokens with state S0 gives the
// closed form of LLM/src/CoreML/MtpRollback.swift:3-12:
//   S_m = e^{G_m} S0 + sum_{s<=m} e^{G_m - G_s} k_s delta_s^T,  G = inclusive
// cumulative sum of g inside the chunk.  Writing delta for all L tokens at once:
//   A[t][s] = beta_t e^{G_t - G_s} (k_t . k_s)        (s < t, else 0)
//   T = (I + A)^-1                                   (unit lower triangular)
//   W = T diag(beta e^G) K,  U = T diag(beta) V,  delta = U - W S0
//   O = qScale (diag(e^G) Q S0) + P delta,  P[t][s] = qScale e^{G_t-G_s} (q_t . k_s), s <= t
//   S_L = e^{G_L} S0 + K^T diag(e^{G_L - G}) delta
// Every exponent is a difference G_t - G_s <= 0 (or G <= 0), so no factor
// exceeds 1 and nothing overflows however long the decay runs.
//
// MI355X design.  Every product above runs on v_mfma_f32_16x16x32_f16 with
// f32 accumulation.  Operands that are f32 -- S, delta, T, beta e^G k,
// beta v, P, and q, k, v themselves when they arrive as f32 -- are split into
// hi = f16(x) and lo = f16(x - hi) and multiplied as hi*hi + hi*lo + lo*hi
// (about 22 significant bits), so the result tracks the f32 recurrence of the
// reference's prefill scan.  f16 q, k, v (BASELINE's prefill inputs) are used
// as they are.
//   gdn_prep  (value head, chunk): K K^T and Q K^T on the matrix cores give A
//             and P; I + A is inverted in 16 x 16 blocks (diagonal blocks by
//             forward substitution, one wave each, then the block below, all
//             256 threads); then W = T X and U = T Y (the UT transform) on the
//             matrix cores.  The chunks are independent.
//   gdn_scan  (value head, 16 columns of S): walks the chunks in order.  One
//             wave is the serial chain: delta = U - W S, S <- e^{G_L} S +
//             K^T (e^{G_L-G} delta), everything it carries in its registers;
//             a second wave forms O = qScale (e^G (Q S) + P delta) beside the
//             next chunk.  Value columns of S are independent, which is what
//             splits the serial part across workgroups.
// Chunks are of 32 tokens whichever chunk length the caller names: the sums
// are the same, and with the kernels built for 64 too, 64 was the slower at
// every shape measured (16 heads, T = 512, f16: 39 us against 30; a 64 x 64
// inverse has three more dependent block levels, and half the units).
// Workspace per (head, chunk) unit, every operand in the order in which the
// scan's lanes load it (one contiguous KiB per load instruction): W hi/lo,
// U, P hi/lo, e^G and e^{G_L-G}; per (key head, chunk) K^T (hi, and lo for
// f32 k) and for f32 q its split.  Rows past a chunk's tokens are zero.
#include "gd_internal.h"

#include <algorithm>

namespace {

constexpr int DK = 128;          // key size handled
constexpr int DV = 128;          // value size handled
constexpr int NCOL = 16;         // value columns of S per scan workgroup
constexpr int CP = 32;           // tokens per chunk
constexpr int PADK = DK + 8;     // LDS row of 128 f16 plus 16 bytes (bank spread)

__device__ __forceinline__ f32x4 mfma(const f16x8 &a, const f16x8 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// gd_split_f16 of eight values.
__device__ __forceinline__ void split8(const float (&x)[8], f16x8 &hi, f16x8 &lo) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        f16x2 h, l;
        gd_split2_f16(x[e], x[e + 1], h, l);
        hi[e] = h[0];
        hi[e + 1] = h[1];
        lo[e] = l[0];
        lo[e + 1] = l[1];
    }
}

// hi*hi + hi*lo + lo*hi, accumulated into c.
__device__ __forceinline__ f32x4 mfma3(const f16x8 &ah, const f16x8 &al, const f16x8 &bh,
                                       const f16x8 &bl, f32x4 c) {
    c = mfma(ah, bh, c);
    c = mfma(ah, bl, c);
    return mfma(al, bh, c);
}

// Eight consecutive activations as loaded (f16 or f32), converted by cvt8:
// keeping them raw lets a prefetch stay in flight until the values are used.
template <typename IO> struct Raw8;
template <> struct Raw8<uint16_t> { u32x4 v; };
template <> struct Raw8<float> { f32x4 a, b; };
template <typename IO>
__device__ __forceinline__ Raw8<IO> load_raw8(const void *base, int64_t idx) {
    Raw8<IO> r;
    if constexpr (sizeof(IO) == 2) {
        r.v = *(const u32x4 *)((const uint16_t *)base + idx);
    } else {
        const f32x4 *p = (const f32x4 *)((const float *)base + idx);
        r.a = p[0];
        r.b = p[1];
    }
    return r;
}
// As f16, zero when !ok.
template <typename IO>
__device__ __forceinline__ f16x8 cvt8(const Raw8<IO> &r, bool ok) {
    f16x8 h;
    if constexpr (sizeof(IO) == 2) {
        h = __builtin_bit_cast(f16x8, ok ? r.v : u32x4{0, 0, 0, 0});
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            h[e] = ok ? (f16)r.a[e] : (f16)0.0f;
            h[4 + e] = ok ? (f16)r.b[e] : (f16)0.0f;
        }
    }
    return h;
}

// hi/lo split of the eight f32 values of a raw load (zeros when !ok).
template <typename IO>
__device__ __forceinline__ void split_raw8(const Raw8<IO> &r, bool ok, f16x8 &hi, f16x8 &lo) {
    float x[8];
    if constexpr (sizeof(IO) == 4) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            x[e] = ok ? r.a[e] : 0.f;
            x[4 + e] = ok ? r.b[e] : 0.f;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = 0.f;      // not used for f16 inputs
    }
    split8(x, hi, lo);
}

// A 16 x 32 (or 32 x 16) operand of the 16x16x32 MFMA as one "fragment": 64
// lanes x 8 f16 (lane lr + 16 g: row or column lr, K positions 8g .. 8g + 7).
// The rows of a pair of accumulator tiles stand for keys (or tokens) in such
// an order that the eight values a lane holds of the pair, rows 4g .. 4g + 3
// of each, are elements 8g .. 8g + 7: row 4a + b of tile q is element perm(q,
// 4a + b) = 8a + 4q + b of the pair's 32.  A result in accumulators (S,
// delta) is then the next product's operand, K positions in natural order,
// without leaving its lane.
__device__ __forceinline__ int perm(int q, int r) { return 8 * (r >> 2) + 4 * q + (r & 3); }

struct Work {
    f16 *Wh, *Wl;     // [u][2 token tiles (perm)][4 key groups][64][8]: -W
    float *U;         // [u][8 column tiles][2 token tiles (perm)][64][4]
    f16 *Ph, *Pl;     // [u][2 token tiles][64][8] (K: tokens s)
    f16 *KT;          // [unit of the key head][8 key tiles (perm by pair)][64][8] (K: tokens)
    f16 *KTl;         // the same, f32 k only: k - f16(k)
    float *G;         // [u][2][CP]: e^G, e^{G_L - G}
    // f32 q only, [unit of the key head][2 token tiles][4 key groups][64][8]:
    // q split (the scan's output wave reading and splitting f32 rows itself
    // took the scan from 17.4 to 19.1 us, 16 heads, T = 512).
    f16 *Qh, *Ql;
};
constexpr size_t WFRAG = 2 * 4 * 64 * 8, UFRAG = 8 * 2 * 64 * 4, PFRAG = 2 * 64 * 8, KFRAG = 8 * 64 * 8;

struct PrepArgs {
    const void *q, *k, *v;
    int64_t q_stride, k_stride, v_stride;
    const float *g, *beta;
    Work w;
    int64_t T;
    int nV, nK, nchunks;
};

template <typename IO>
__global__ __launch_bounds__(256) void gdn_prep(PrepArgs a) {
    // f32 q, k, v: hi/lo pairs.  The lo halves of K and Q are needed only
    // until A and P are formed, so they share the space of Xh and Xl, which
    // are first written after that (and X, Y are then formed from the f32
    // inputs themselves, re-read from L2).
    constexpr bool HL = sizeof(IO) == 4;
    __shared__ __attribute__((aligned(16))) f16 Ks[CP][PADK];
    __shared__ __attribute__((aligned(16))) f16 QVs[CP][PADK];     // Q, later V
    __shared__ __attribute__((aligned(16))) f16 Xh[DK][CP + 8], Xl[DK][CP + 8];
    __shared__ __attribute__((aligned(16))) f16 Yh[DV][CP + 8], Yl[DV][CP + 8];
    static_assert(sizeof(Xh) >= sizeof(Ks), "K lo must fit where Xh lives");
    f16 (*Kl)[PADK] = reinterpret_cast<f16 (*)[PADK]>(&Xh[0][0]);
    f16 (*Ql)[PADK] = reinterpret_cast<f16 (*)[PADK]>(&Xl[0][0]);
    __shared__ __attribute__((aligned(16))) float Af[CP][CP + 4];
    __shared__ __attribute__((aligned(16))) float Tf[CP][CP + 4];
    __shared__ __attribute__((aligned(16))) float Ms[(CP / 16 - 1) * 256];   // block products
    __shared__ float Gs[CP], Bs[CP], BEs[CP];               // G, beta, beta e^G

    // Workgroup b runs on XCD b % 8.  When the units divide by 8, XCD x takes
    // the contiguous units x * units/8 .., so a head's chunks are written into
    // the L2 of the XCD whose scan workgroups read them (the scan deals each
    // head's column slices to one XCD in the same order).
    const int units = (int)gridDim.x;
    const int ub = units % 8 == 0 ? (int)((blockIdx.x & 7) * (units >> 3) + (blockIdx.x >> 3))
                                  : (int)blockIdx.x;
    const int hv = ub / a.nchunks, c = ub % a.nchunks;
    const int hk = hv % a.nK;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t t0 = (int64_t)c * CP;
    const int L = (int)min((int64_t)CP, a.T - t0);
    const int64_t u = (int64_t)hv * a.nchunks + c;
    // K^T and Q do not depend on the value head: the first of a key head
    // writes them.
    const bool first = hv == hk;
    const int lr = lane & 15, kg = lane >> 4;

    // Rows of K and Q (and V, kept in registers until Q is done): thread e
    // handles 8 consecutive elements of row e / 16.
    // Every load goes out before any is converted (rows past the chunk read
    // token 0 and are zeroed at conversion): loads under a branch, converted
    // on arrival, waited for one by one.
    constexpr int NE = CP * DK / 8 / 256;                   // entries per thread
    f16x8 vreg[NE];
    Raw8<IO> rk[NE], rq[NE], rv[NE];
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + 256 * n, t = e >> 4, i8 = (e & 15) * 8;
        const int64_t tok = t0 + (t < L ? t : 0);
        rk[n] = load_raw8<IO>(a.k, tok * a.k_stride + (int64_t)hk * DK + i8);
        rq[n] = load_raw8<IO>(a.q, tok * a.q_stride + (int64_t)hk * DK + i8);
        rv[n] = load_raw8<IO>(a.v, tok * a.v_stride + (int64_t)hv * DV + i8);
    }
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + 256 * n, t = e >> 4, i8 = (e & 15) * 8;
        const bool ok = t < L;
        if constexpr (HL) {
            f16x8 h, l;
            split_raw8<IO>(rk[n], ok, h, l);
            *(f16x8 *)&Ks[t][i8] = h;
            *(f16x8 *)&Kl[t][i8] = l;
            split_raw8<IO>(rq[n], ok, h, l);
            *(f16x8 *)&QVs[t][i8] = h;
            *(f16x8 *)&Ql[t][i8] = l;
            if (first) {                                      // rows past the chunk: zeros
                const size_t qi = u * WFRAG + (((t >> 4) * 4 + (i8 >> 5)) * 64 + ((i8 >> 3) & 3) * 16 + (t & 15)) * 8;
                *(f16x8 *)&a.w.Qh[qi] = h;
                *(f16x8 *)&a.w.Ql[qi] = l;
            }
        } else {
            *(f16x8 *)&Ks[t][i8] = cvt8<IO>(rk[n], ok);
            *(f16x8 *)&QVs[t][i8] = cvt8<IO>(rq[n], ok);
            vreg[n] = cvt8<IO>(rv[n], ok);
        }
    }
    if (wave == 0) {
        // Inclusive cumulative gate inside the chunk (wave prefix sum); rows
        // past L keep G[L-1] and get beta = 0.
        float gv = lane < L ? a.g[(t0 + lane) * a.nV + hv] : 0.f;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float o = __shfl_up(gv, off, 64);
            if (lane >= off) gv += o;
        }
        if (lane < CP) {
            const float bt = lane < L ? a.beta[(t0 + lane) * a.nV + hv] : 0.f;
            Gs[lane] = gv;
            Bs[lane] = bt;
            BEs[lane] = bt * __expf(gv);
        }
    }
    __syncthreads();

    // K K^T -> A (s < t) and (Q K^T)^T -> P (s <= t), lower tiles on the matrix
    // cores; P's upper tiles are written as zeros.  A has rows t in the
    // accumulators' rows; P has them in its columns, so that a lane holds four
    // consecutive s of one t.
    constexpr int NB = CP / 16;
    // Unrolled: a wave's tiles are independent, so their LDS reads, MFMA
    // chains and stores can overlap.
#pragma unroll
    for (int tile = wave; tile < 2 * NB * NB; tile += 4) {
        const bool isP = tile >= NB * NB;
        const int tt = isP ? tile - NB * NB : tile;
        const int ti = tt / NB, si = tt % NB;
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        if (si <= ti) {
#pragma unroll
            for (int k0 = 0; k0 < DK; k0 += 32) {
                const f16x8 tv = isP ? *(const f16x8 *)&QVs[ti * 16 + lr][k0 + kg * 8]
                                     : *(const f16x8 *)&Ks[ti * 16 + lr][k0 + kg * 8];
                const f16x8 sv = *(const f16x8 *)&Ks[si * 16 + lr][k0 + kg * 8];
                if constexpr (HL) {
                    const f16x8 tl = isP ? *(const f16x8 *)&Ql[ti * 16 + lr][k0 + kg * 8]
                                         : *(const f16x8 *)&Kl[ti * 16 + lr][k0 + kg * 8];
                    const f16x8 sl = *(const f16x8 *)&Kl[si * 16 + lr][k0 + kg * 8];
                    acc = isP ? mfma3(sv, sl, tv, tl, acc) : mfma3(tv, tl, sv, sl, acc);
                } else {
                    acc = isP ? mfma(sv, tv, acc) : mfma(tv, sv, acc);
                }
            }
        }
        f16x4 ph, pl;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = kg * 4 + v;                         // accumulator row
            const int t = ti * 16 + (isP ? lr : r), s = si * 16 + (isP ? r : lr);
            const float dec = __expf(Gs[t] - Gs[s]);          // factor in (0, 1]
            if (!isP) {
                Af[t][s] = (s < t && t < L) ? Bs[t] * dec * acc[v] : 0.f;
            } else {
                const float p = (s <= t && t < L) ? dec * acc[v] : 0.f;
                f16 h, l;
                gd_split_f16(p, h, l);
                ph[v] = h;
                pl[v] = l;
            }
        }
        if (isP) {
            // s = 16 si + 4 kg + v of token row lr: lane group s / 8.
            const size_t pi = u * PFRAG + (ti * 64 + (2 * si + (kg >> 1)) * 16 + lr) * 8 + 4 * (kg & 1);
            *(f16x4 *)&a.w.Ph[pi] = ph;
            *(f16x4 *)&a.w.Pl[pi] = pl;
        }
    }
    __syncthreads();
    // V replaces Q (f16 inputs; f32 ones are re-read for Y below).
    if constexpr (!HL) {
#pragma unroll
        for (int n = 0; n < NE; n++) {
            const int e = tid + 256 * n, t = e >> 4, i8 = (e & 15) * 8;
            *(f16x8 *)&QVs[t][i8] = vreg[n];
        }
    }
    __syncthreads();

    // T = (I + A)^-1 in 16 x 16 blocks (A is strictly lower triangular).
    // Diagonal blocks first, wave w inverting block w by forward
    // substitution with lane s < 16 holding its column s: T[t][s] =
    // -sum_{m<t} A[t][m] T[m][s] (T[m][s] = 0 for m < s, T[s][s] = 1);
    // blocks above the diagonal are zero.
    if (wave < NB && lane < 16) {
        const int b0 = wave * 16, s = lane;
        float Tc[16];
#pragma unroll
        for (int m = 0; m < 16; m++) Tc[m] = m == s ? 1.f : 0.f;
#pragma unroll
        for (int t = 1; t < 16; t++) {
            float acc = 0.f;
#pragma unroll
            for (int m = 0; m < t; m++) acc = fmaf(Af[b0 + t][b0 + m], Tc[m], acc);
            Tc[t] = t == s ? 1.f : -acc;
        }
#pragma unroll
        for (int m = 0; m < 16; m++) Tf[b0 + m][b0 + s] = Tc[m];
    }
    for (int e = tid; e < CP * CP; e += 256) {
        const int r = e / CP, cc = e % CP;
        if ((cc >> 4) > (r >> 4)) Tf[r][cc] = 0.f;
    }
    __syncthreads();
    // Blocks below the diagonal by distance d = i - j, each level from the
    // ones before it: T_ij = -T_ii (sum_{k=j}^{i-1} A_ik T_kj).  Thread e
    // takes element (r, cc) of block i = d + e / 256.
    for (int d = 1; d < NB; d++) {
        for (int e = tid; e < (NB - d) * 256; e += 256) {
            const int i = d + (e >> 8), j = i - d, r = (e >> 4) & 15, cc = e & 15;
            float m = 0.f;
            for (int k = j; k < i; k++)
#pragma unroll
                for (int q = 0; q < 16; q++)
                    m = fmaf(Af[i * 16 + r][k * 16 + q], Tf[k * 16 + q][j * 16 + cc], m);
            Ms[e] = m;
        }
        __syncthreads();
        for (int e = tid; e < (NB - d) * 256; e += 256) {
            const int i = d + (e >> 8), j = i - d, r = (e >> 4) & 15, cc = e & 15;
            const float *mb = Ms + (e & ~255);
            float t = 0.f;
#pragma unroll
            for (int q = 0; q < 16; q++) t = fmaf(Tf[i * 16 + r][i * 16 + q], mb[q * 16 + cc], t);
            Tf[i * 16 + r][j * 16 + cc] = -t;
        }
        __syncthreads();
    }
    // X^T = (diag(beta e^G) K)^T and Y^T = (diag(beta) V)^T, split, as the
    // operands of T X and T Y, and K^T to the workspace for the scan's
    // state update (its A operand): entry (lane group g, i) takes tokens
    // 8g .. 8g + 7, lanes along i so that the row reads of K and V hit
    // distinct banks.
    // f32 inputs: k and v come from global memory (the chunk was read moments
    // ago, so from L2), every load of an entry issued before any is used, at
    // clamped rows (rows past the chunk are zeroed on use).
    for (int e = tid; e < DK * (CP / 8); e += 256) {
        const int g = e / DK, i = e % DK;
        float xv[8], yv[8];
        f16x8 kv, kl;
        if constexpr (HL) {
            float kf[8], vf[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int64_t tok = t0 + (8 * g + q < L ? 8 * g + q : 0);
                kf[q] = ((const float *)a.k)[tok * a.k_stride + (int64_t)hk * DK + i];
                vf[q] = ((const float *)a.v)[tok * a.v_stride + (int64_t)hv * DV + i];
            }
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int s = 8 * g + q;
                const float kk = s < L ? kf[q] : 0.f, vv = s < L ? vf[q] : 0.f;
                f16 kh, kt;
                gd_split_f16(kk, kh, kt);
                kv[q] = kh;
                kl[q] = kt;
                xv[q] = BEs[s] * kk;
                yv[q] = Bs[s] * vv;
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int s = 8 * g + q;
                kv[q] = Ks[s][i];
                xv[q] = BEs[s] * (float)kv[q];
                yv[q] = Bs[s] * (float)QVs[s][i];
            }
        }
        f16x8 h, l;
        split8(xv, h, l);
        *(f16x8 *)&Xh[i][8 * g] = h;
        *(f16x8 *)&Xl[i][8 * g] = l;
        split8(yv, h, l);
        *(f16x8 *)&Yh[i][8 * g] = h;
        *(f16x8 *)&Yl[i][8 * g] = l;
        // Key i is row 4a + b of tile q of its pair: i = 32 p + 8 a + 4 q + b.
        const int kt = 2 * (i >> 5) + ((i >> 2) & 1), kr = 4 * ((i >> 3) & 3) + (i & 3);
        const size_t ki = u * KFRAG + (kt * 64 + g * 16 + kr) * 8;
        if (first) {
            *(f16x8 *)&a.w.KT[ki] = kv;
            if constexpr (HL) *(f16x8 *)&a.w.KTl[ki] = kl;
        }
    }
    if (tid < CP) {
        a.w.G[(size_t)u * 2 * CP + tid] = expf(Gs[tid]);
        a.w.G[(size_t)u * 2 * CP + CP + tid] = expf(Gs[CP - 1] - Gs[tid]);
    }
    __syncthreads();

    // -W = -T X and U = T Y: wave w takes the token tile rb = w % 2 (perm) and
    // four column tiles of each.  W goes out with tokens in the accumulators'
    // columns, so a lane holds the eight keys of a fragment; U with tokens in
    // their rows, as the scan's delta.
    const int rb = wave & 1, half = wave >> 1;
    f16x8 th, tl;
    {
        float tv[8];
#pragma unroll
        for (int q = 0; q < 8; q++) tv[q] = Tf[perm(rb, lr)][kg * 8 + q];
        split8(tv, th, tl);
    }
    auto operand = [&](const f16 (*src)[CP + 8], int row) { return *(const f16x8 *)&src[row][kg * 8]; };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int p = 2 * half + j;                          // key group
        f16x8 h, l;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int key = 32 * p + perm(q, lr);
            const f32x4 acc = mfma3(operand(Xh, key), operand(Xl, key), th, tl, zero);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                f16 hh, ll;
                gd_split_f16(-acc[v], hh, ll);
                h[4 * q + v] = hh;
                l[4 * q + v] = ll;
            }
        }
        const size_t wi = u * WFRAG + ((rb * 4 + p) * 64 + lane) * 8;
        *(f16x8 *)&a.w.Wh[wi] = h;
        *(f16x8 *)&a.w.Wl[wi] = l;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int ct = 4 * half + j;
        const f32x4 acc = mfma3(th, tl, operand(Yh, ct * 16 + lr), operand(Yl, ct * 16 + lr), zero);
        *(f32x4 *)&a.w.U[u * UFRAG + ((ct * 2 + rb) * 64 + lane) * 4] = acc;
    }
}

struct ScanArgs {
    const void *q;
    int64_t q_stride;
    Work w;
    float *S;
    void *o;
    int64_t o_stride;
    int64_t T;
    int nV, nK, nchunks;
    float qScale;
};

// The scan's workgroup is two waves.  The chain wave walks the recurrence and
// is what its time is made of: per chunk delta = U - W S, then S <- e^{G_L} S
// + K^T (e^{G_L-G} delta).  Its 128 keys x 16 columns of S sit in eight
// accumulator tiles; their hi/lo split is the B operand of W S lane for lane,
// and delta's that of K^T E, so nothing of the chain goes through LDS or
// waits for another wave: 40 (f16 k) or 48 MFMAs and the splits.  The
// output wave computes O = qScale (e^G (Q S) + P delta) of a chunk beside the
// chain's state update and next delta, from the split of S and delta that the
// chain leaves in LDS (by chunk parity: one barrier per chunk).
//   Operands come one contiguous KiB per load, refilled for the next chunk as
// soon as this one has used them.  (Two register sets, two chunks ahead, do
// not fit 256 registers: the accumulators then move through AGPRs, 23.5 us.)
//   16 heads, T = 512 (16 chunks): 15.6 us with f16 inputs, 17.3 with f32 (a
// chain of four waves that exchanged S and delta through LDS, two barriers a
// chunk: 22, at chunks of 64, and 24.4), about 0.8 us a chunk; 48 heads, T =
// 1000, f32: 47 us (107 at chunks of 64).  What bounds it is that chain of
// dependent MFMAs and splits; with more than one slice per CU, the operands
// through the CU's cache (54 KiB a chunk and slice).
constexpr int SCAN_THREADS = 128;     // chain wave, output wave

// The chain's operands of one chunk.
template <bool HL> struct ChainRegs {
    f16x8 wh[2][4], wl[2][4];             // -W by token tile, key group
    f32x4 u[2], ed[2];                    // U and e^{G_L - G} of tokens 8g + 4m + v
    float dec;                            // e^{G_L}
    f16x8 ka[8], kal[HL ? 8 : 1];         // K^T by key tile
};

// Eight f32 in two accumulators -> the operand fragment they make, split.
__device__ __forceinline__ void split_tiles(const f32x4 &x, const f32x4 &y, f16x8 &hi, f16x8 &lo) {
    const float f[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    split8(f, hi, lo);
}

template <typename IO, typename OT>
__global__ __launch_bounds__(SCAN_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_scan(ScanArgs a) {
    constexpr bool HL = sizeof(IO) == 4;
    __shared__ f16x8 Ss[2][2][4][64];     // S of a chunk (parity, hi/lo, key group, lane)
    __shared__ f32x4 Ds[2][2][64];        // delta (parity, token tile, lane)

    constexpr int NCB = DV / NCOL;
    static_assert(NCB % 8 == 0, "the grid must split evenly over the 8 XCDs");
    // Workgroup b runs on XCD b % 8.  The NCB column slices of one head read
    // the same chunk operands (W, P, K^T, Q), so they are dealt to one XCD:
    // slice index (b % 8) * (grid / 8) + b / 8, head that / NCB, so each chunk
    // is fetched into one L2 once instead of into every L2.
    const int sl = (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3));
    const int hv = sl / NCB, ct = sl % NCB, j0 = ct * NCOL;
    const int hk = hv % a.nK;
    const int lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
    // A wave's role as a scalar: the branch below is a jump.
    const bool chain = __builtin_amdgcn_readfirstlane((int)threadIdx.x) < 64;
    auto unit = [&](int c) { return (size_t)hv * a.nchunks + min(c, a.nchunks - 1); };

    if (chain) {
        f32x4 st[8];                      // tile 2p + q: S of keys 32p + 8g + 4q + v, column j0 + lr
        f16x8 sh[4], sl_[4];              // its split by key group
        float *Sg = a.S + (size_t)hv * DK * DV + j0 + lr;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) st[i][v] = Sg[(16 * (i & ~1) + 8 * g + 4 * (i & 1) + v) * DV];
        auto loadW = [&](int c, ChainRegs<HL> &k) {
            const size_t un = unit(c);
            k.dec = a.w.G[un * 2 * CP + CP - 1];
            const f16 *wh = a.w.Wh + un * WFRAG + lane * 8, *wl = a.w.Wl + un * WFRAG + lane * 8;
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    k.wh[m][p] = *(const f16x8 *)(wh + (m * 4 + p) * 512);
                    k.wl[m][p] = *(const f16x8 *)(wl + (m * 4 + p) * 512);
                }
#pragma unroll
            for (int m = 0; m < 2; m++) {
                k.u[m] = *(const f32x4 *)(a.w.U + un * UFRAG + ((ct * 2 + m) * 64 + lane) * 4);
                k.ed[m] = *(const f32x4 *)(a.w.G + un * 2 * CP + CP + 8 * g + 4 * m);
            }
        };
        auto loadK = [&](int c, ChainRegs<HL> &k) {
            const size_t un = (size_t)hk * a.nchunks + min(c, a.nchunks - 1);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                k.ka[i] = *(const f16x8 *)(a.w.KT + un * KFRAG + (i * 64 + lane) * 8);
                if constexpr (HL) k.kal[i] = *(const f16x8 *)(a.w.KTl + un * KFRAG + (i * 64 + lane) * 8);
            }
        };
        auto chunk = [&](int c, ChainRegs<HL> &k) {
            const int b = c & 1;
            // delta = U - W S: hi * hi from U on, the cross terms beside it.
            f32x4 d[2], x[2], y[2];
#pragma unroll
            for (int m = 0; m < 2; m++) {
                d[m] = k.u[m];
                x[m] = y[m] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int p = 0; p < 4; p++) {
                Ss[b][0][p][lane] = sh[p];
                Ss[b][1][p][lane] = sl_[p];
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    d[m] = mfma(k.wh[m][p], sh[p], d[m]);
                    x[m] = mfma(k.wh[m][p], sl_[p], x[m]);
                    y[m] = mfma(k.wl[m][p], sh[p], y[m]);
                }
            }
            f32x4 e[2];
#pragma unroll
            for (int m = 0; m < 2; m++) {
                d[m] += x[m] + y[m];
                Ds[b][m][lane] = d[m];
                e[m] = k.ed[m] * d[m];
            }
            f16x8 eh, el;
            split_tiles(e[0], e[1], eh, el);
            const float dec = k.dec;
            // (Fenced: the compiler would sink the loads next to their use.)
            __builtin_amdgcn_sched_barrier(0);
            loadW(c + 1, k);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            // S <- e^{G_L} S + K^T E, and its split as the pairs of tiles finish.
#pragma unroll
            for (int p = 0; p < 4; p++) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int i = 2 * p + q;
                    f32x4 acc = mfma(k.ka[i], eh, st[i] * dec);
                    acc = mfma(k.ka[i], el, acc);
                    if constexpr (HL) acc = mfma(k.kal[i], eh, acc);
                    st[i] = acc;
                }
                split_tiles(st[2 * p], st[2 * p + 1], sh[p], sl_[p]);
            }
            __builtin_amdgcn_sched_barrier(0);
            loadK(c + 1, k);
            __builtin_amdgcn_sched_barrier(0);
        };
        ChainRegs<HL> k;
        // In the loop's order, so that its wait counts are exact.
        __builtin_amdgcn_sched_barrier(0);
        loadW(0, k);
        __builtin_amdgcn_sched_barrier(0);
        loadK(0, k);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 4; p++) split_tiles(st[2 * p], st[2 * p + 1], sh[p], sl_[p]);
        for (int c = 0; c < a.nchunks; c++) chunk(c, k);
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) Sg[(16 * (i & ~1) + 8 * g + 4 * (i & 1) + v) * DV] = st[i][v];
    } else {
        // Q (f16 as it is, f32 as the split prep stored), P and e^G of tokens
        // 16 m + lr: refilled for the next chunk as soon as they are used.
        f16x8 qh[2][4], ql[HL ? 2 : 1][4], ph[2], pl[2];
        float eg[2];
        // Vector stores where every row keeps their alignment.
        const bool vec = ((uintptr_t)a.o % (4 * sizeof(OT))) == 0 && a.o_stride % 4 == 0;
        auto loadQ = [&](int c) {
            const size_t un = (size_t)hk * a.nchunks + min(c, a.nchunks - 1);
            const int64_t t0 = (int64_t)min(c, a.nchunks - 1) * CP;
            const int L = (int)min((int64_t)CP, a.T - t0);
#pragma unroll
            for (int m = 0; m < 2; m++)
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    if constexpr (HL) {
                        qh[m][p] = *(const f16x8 *)(a.w.Qh + un * WFRAG + ((m * 4 + p) * 64 + lane) * 8);
                        ql[m][p] = *(const f16x8 *)(a.w.Ql + un * WFRAG + ((m * 4 + p) * 64 + lane) * 8);
                    } else {
                        // Rows past the chunk: its last token's (not stored).
                        qh[m][p] = *(const f16x8 *)((const uint16_t *)a.q + (t0 + min(16 * m + lr, L - 1)) * a.q_stride +
                                                    (int64_t)hk * DK + 32 * p + 8 * g);
                    }
                }
        };
        auto loadP = [&](int c) {
            const size_t un = unit(c);
#pragma unroll
            for (int m = 0; m < 2; m++) {
                eg[m] = a.w.G[un * 2 * CP + 16 * m + lr];
                ph[m] = *(const f16x8 *)(a.w.Ph + un * PFRAG + (m * 64 + lane) * 8);
                pl[m] = *(const f16x8 *)(a.w.Pl + un * PFRAG + (m * 64 + lane) * 8);
            }
        };
        __builtin_amdgcn_sched_barrier(0);
        loadQ(0);
        __builtin_amdgcn_sched_barrier(0);
        loadP(0);
        __builtin_amdgcn_sched_barrier(0);
        for (int c = 0; c < a.nchunks; c++) {
            const int b = c & 1;
            __syncthreads();
            // O^T: value columns in the accumulators' rows (S and delta as A
            // operands), tokens in their columns, so a lane stores four
            // consecutive columns of one token.
            f32x4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const f16x8 sh = Ss[b][0][p][lane], sl_ = Ss[b][1][p][lane];
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    o[m] = mfma(sh, qh[m][p], o[m]);
                    o[m] = mfma(sl_, qh[m][p], o[m]);
                    if constexpr (HL) o[m] = mfma(sh, ql[m][p], o[m]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            loadQ(c + 1);
            __builtin_amdgcn_sched_barrier(0);
            f16x8 dh, dl;
            split_tiles(Ds[b][0][lane], Ds[b][1][lane], dh, dl);
            const int64_t t0 = (int64_t)c * CP;
            const int L = (int)min((int64_t)CP, a.T - t0);
            // Rows t >= L lie past the bounds-checked resource: not stored.
            const __amdgpu_buffer_rsrc_t ors = gd_rsrc((OT *)a.o + t0 * a.o_stride,
                                                       (uint32_t)L * (uint32_t)a.o_stride * sizeof(OT));
#pragma unroll
            for (int m = 0; m < 2; m++) {
                f32x4 acc = o[m] * eg[m];
                acc = mfma3(dh, dl, ph[m], pl[m], acc);
                acc *= a.qScale;
                const uint32_t oo = ((uint32_t)(16 * m + lr) * (uint32_t)a.o_stride + (uint32_t)hv * DV +
                                     j0 + 4 * g) * sizeof(OT);
                if constexpr (sizeof(OT) == 4) {
                    if (vec) {
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), ors, oo, 0, 0);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[v]), ors, oo + 4 * v, 0, 0);
                    }
                } else {
                    if (vec) {
                        const u32x2 w = {(uint32_t)gd_f2h(acc[0]) | ((uint32_t)gd_f2h(acc[1]) << 16),
                                         (uint32_t)gd_f2h(acc[2]) | ((uint32_t)gd_f2h(acc[3]) << 16)};
                        __builtin_amdgcn_raw_buffer_store_b64(w, ors, oo, 0, 0);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            __builtin_amdgcn_raw_buffer_store_b16(gd_f2h(acc[v]), ors, oo + 2 * v, 0, 0);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            loadP(c + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

int launch(gd_ctx *ctx, const PrepArgs &pa, const ScanArgs &sa, int io_dtype, int o_dtype) {
    const unsigned units = (unsigned)(pa.nV * pa.nchunks);
    if (io_dtype == GD_F32)
        hipLaunchKernelGGL((gdn_prep<float>), dim3(units), dim3(256), 0, ctx->stream, pa);
    else
        hipLaunchKernelGGL((gdn_prep<uint16_t>), dim3(units), dim3(256), 0, ctx->stream, pa);
    GD_LAUNCHED(ctx, "gdn_prep");
    const dim3 grid((unsigned)(sa.nV * (DV / NCOL)));
#define GD_SCAN(IO, OT) \
    hipLaunchKernelGGL((gdn_scan<IO, OT>), grid, dim3(SCAN_THREADS), 0, ctx->stream, sa)
    if (io_dtype == GD_F32) { if (o_dtype == GD_F32) GD_SCAN(float, float); else GD_SCAN(float, uint16_t); }
    else { if (o_dtype == GD_F32) GD_SCAN(uint16_t, float); else GD_SCAN(uint16_t, uint16_t); }
#undef GD_SCAN
    GD_LAUNCHED(ctx, "gdn_scan");
    return GD_OK;
}

}  // namespace

int gd_ctx_workspace(gd_ctx *ctx, size_t bytes, void **out);

namespace {

// Checks the arguments; *bytes receives the scratch the call needs (0 for T = 0).
int prefill_check(gd_ctx *ctx, const char *fn, int64_t T, int nV, int nK, int dk, int dv,
                  const void *q, int64_t q_stride, const void *k, int64_t k_stride,
                  const void *v, int64_t v_stride, int io_dtype, const float *g,
                  const float *beta, float *S, void *o, int64_t o_stride, int o_dtype, int C,
                  size_t *bytes) {
    GD_REQUIRE(ctx, q && k && v && g && beta && S && o, "%s: null pointer", fn);
    GD_REQUIRE(ctx, dk == DK && dv == DV, "%s: dk=%d dv=%d (takes 128/128)", fn, dk, dv);
    GD_REQUIRE(ctx, C == 16 || C == 32 || C == 64, "%s: chunk %d not 16/32/64", fn, C);
    GD_REQUIRE(ctx, nV > 0 && nK > 0 && T >= 0, "%s: nV=%d nK=%d T=%lld", fn, nV, nK,
               (long long)T);
    GD_REQUIRE(ctx, io_dtype == GD_F32 || io_dtype == GD_F16, "%s: bad io dtype", fn);
    GD_REQUIRE(ctx, o_dtype == GD_F32 || o_dtype == GD_F16, "%s: bad o dtype", fn);
    GD_REQUIRE(ctx, q_stride >= (int64_t)nK * dk && k_stride >= (int64_t)nK * dk &&
                        v_stride >= (int64_t)nV * dv && o_stride >= (int64_t)nV * dv,
               "%s: strides smaller than a token row", fn);
    // A chunk's output rows are stored through one 32-bit buffer range.
    GD_REQUIRE(ctx, o_stride <= (1 << 24), "%s: o_stride %lld above 2^24", fn,
               (long long)o_stride);
    // Rows are read 8 elements at a time.
    const int vec = io_dtype == GD_F16 ? 8 : 4;
    const int esz = io_dtype == GD_F16 ? 2 : 4;
    GD_REQUIRE(ctx, q_stride % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 &&
                        ((uintptr_t)q % (vec * esz)) == 0 && ((uintptr_t)k % (vec * esz)) == 0 &&
                        ((uintptr_t)v % (vec * esz)) == 0,
               "%s: q/k/v rows must be 8-element strided and %d-byte aligned", fn, vec * esz);
    *bytes = 0;
    if (T == 0) return GD_OK;
    // The documented need (the allocation-free entry's limit): per chunk of the
    // caller's C tokens, of which the kernels' own (prefill_bytes) is a little
    // more at C = 32 (the second decay factor) and less otherwise.
    const size_t units = (size_t)nV * (size_t)((T + C - 1) / C);
    const size_t R = C < 32 ? 32 : C;
    const size_t nkt = io_dtype == GD_F32 ? 2 : 1;
    *bytes = units * (2 * R * DK * 2 + R * DV * 4 + 2 * R * R * 2 + nkt * DK * R * 2 +
                      R * 4 + (nkt - 1) * 2 * R * DK * 2);
    return GD_OK;
}

// Workspace of T tokens: the layout prefill_run carves.
size_t prefill_bytes(int64_t T, int nV, int nK, int io_dtype) {
    const size_t units = (size_t)nV * (size_t)((T + CP - 1) / CP);
    const size_t kunits = units / nV * std::min(nV, nK);
    return units * (2 * WFRAG * 2 + UFRAG * 4 + 2 * PFRAG * 2 + 2 * CP * 4) +
           kunits * (io_dtype == GD_F32 ? 2 * KFRAG + 2 * WFRAG : KFRAG) * 2;
}

// Launches prep + scan with their per-(head, chunk) operands in ws (at least
// prefill_bytes).  Every byte of ws the scan reads is written by prep in the
// same call, so ws needs no clearing.
int prefill_run(gd_ctx *ctx, void *ws, int64_t T, int nV, int nK, const void *q,
                int64_t q_stride, const void *k, int64_t k_stride, const void *v,
                int64_t v_stride, int io_dtype, const float *g, const float *beta, float *S,
                void *o, int64_t o_stride, int o_dtype, float qScale) {
    const int nchunks = (int)((T + CP - 1) / CP);
    const size_t units = (size_t)nV * nchunks;
    const bool hl = io_dtype == GD_F32;
    uint8_t *p = (uint8_t *)ws;
    auto take = [&](size_t bytes) { uint8_t *r = p; p += bytes; return r; };
    Work w{};
    w.Wh = (f16 *)take(units * WFRAG * 2);
    w.Wl = (f16 *)take(units * WFRAG * 2);
    w.U = (float *)take(units * UFRAG * 4);
    w.Ph = (f16 *)take(units * PFRAG * 2);
    w.Pl = (f16 *)take(units * PFRAG * 2);
    const size_t kunits = (size_t)std::min(nV, nK) * nchunks;
    w.KT = (f16 *)take(kunits * KFRAG * 2);
    if (hl) w.KTl = (f16 *)take(kunits * KFRAG * 2);
    w.G = (float *)take(units * 2 * CP * 4);
    if (hl) w.Qh = (f16 *)take(kunits * WFRAG * 2);
    if (hl) w.Ql = (f16 *)take(kunits * WFRAG * 2);

    PrepArgs pa{q, k, v, q_stride, k_stride, v_stride, g, beta, w, T, nV, nK, nchunks};
    ScanArgs sa{q, q_stride, w, S, o, o_stride, T, nV, nK, nchunks, qScale};
    return launch(ctx, pa, sa, io_dtype, o_dtype);
}

// Scratch of gd_gdn_prefill_noalloc: a file-scope device array, so the entry
// needs no allocation.  Each device holds its own copy until the process
// ends; host code reaches it only through the address hipGetSymbolAddress
// returns for the current device (kept per context), never through the
// array's name.  Every call on a device shares it.
// Shapes are admitted by the documented GD_GDN_PREFILL_SCRATCH_BYTES at the
// documented bytes per chunk; the kernels' second decay factor (128 bytes a
// unit, at most 742 units admitted at C = 32) comes on top.
constexpr size_t PREFILL_SCRATCH_BYTES = GD_GDN_PREFILL_SCRATCH_BYTES;
constexpr size_t PREFILL_SCRATCH_EXTRA = 1u << 18;
static __device__ __align__(256) unsigned char scratch[PREFILL_SCRATCH_BYTES + PREFILL_SCRATCH_EXTRA];

}  // namespace

int gd_prefill_scratch_attach(gd_ctx *ctx) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) {
        ctx->prefill_scratch = nullptr;
        return gd_hip_fail(ctx, e, "prefill scratch: hipGetSymbolAddress");
    }
    ctx->prefill_scratch = p;
    return GD_OK;
}

extern "C" int gd_gdn_prefill(gd_ctx *ctx, int64_t T, int nV, int nK, int dk, int dv,
                              const void *q, int64_t q_stride, const void *k, int64_t k_stride,
                              const void *v, int64_t v_stride, int io_dtype, const float *g,
                              const float *beta, float *S, void *o, int64_t o_stride,
                              int o_dtype, float qScale, int C) {
    GD_CHECK_CTX(ctx);
    size_t bytes = 0;
    int rc = prefill_check(ctx, "gd_gdn_prefill", T, nV, nK, dk, dv, q, q_stride, k, k_stride, v,
                           v_stride, io_dtype, g, beta, S, o, o_stride, o_dtype, C, &bytes);
    if (rc || T == 0) return rc;
    void *ws = nullptr;
    if ((rc = gd_ctx_workspace(ctx, prefill_bytes(T, nV, nK, io_dtype), &ws))) return rc;
    return prefill_run(ctx, ws, T, nV, nK, q, q_stride, k, k_stride, v, v_stride, io_dtype, g,
                       beta, S, o, o_stride, o_dtype, qScale);
}

extern "C" int gd_gdn_prefill_noalloc(gd_ctx *ctx, int64_t T, int nV, int nK, int dk, int dv,
                                      const void *q, int64_t q_stride, const void *k,
                                      int64_t k_stride, const void *v, int64_t v_stride,
                                      int io_dtype, const float *g, const float *beta, float *S,
                                      void *o, int64_t o_stride, int o_dtype, float qScale,
                                      int C) {
    GD_CHECK_CTX(ctx);
    size_t bytes = 0;
    int rc = prefill_check(ctx, "gd_gdn_prefill_noalloc", T, nV, nK, dk, dv, q, q_stride, k,
                           k_stride, v, v_stride, io_dtype, g, beta, S, o, o_stride, o_dtype, C,
                           &bytes);
    if (rc || T == 0) return rc;
    GD_REQUIRE(ctx, bytes <= PREFILL_SCRATCH_BYTES,
               "gd_gdn_prefill_noalloc: needs %zu bytes of scratch for nV=%d x %lld chunks of "
               "%d, above its fixed %zu (GD_GDN_PREFILL_SCRATCH_BYTES); split T or use "
               "gd_gdn_prefill", bytes, nV, (long long)((T + C - 1) / C), C,
               PREFILL_SCRATCH_BYTES);
    GD_REQUIRE(ctx, ctx->prefill_scratch != nullptr,
               "gd_gdn_prefill_noalloc: the scratch array's device address could not be "
               "looked up when the context was created");
    return prefill_run(ctx, ctx->prefill_scratch, T, nV, nK, q, q_stride, k, k_stride, v,
                       v_stride, io_dtype, g, beta, S, o, o_stride, o_dtype, qScale);
}

extern "C" int gd_gdn_scan_batch(gd_ctx *ctx, const float *convOutN, int keyDim, int valueDim,
                                 int convDim, const float *gN, const float *betaN, float *S,
                                 float *oN, int nV, int nK, int dS, float qScale, int64_t N) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, convOutN && gN && betaN && S && oN, "gd_gdn_scan_batch: null pointer");
    GD_REQUIRE(ctx, keyDim == nK * dS && valueDim == nV * dS && convDim >= 2 * keyDim + valueDim,
               "gd_gdn_scan_batch: keyDim/valueDim/convDim inconsistent with nK, nV, dS");
    // The chunked prefill holds 128 x 128 states; other sizes take the
    // token-serial scan, as MetalEnc.gdnScanBatch falls back to
    // gdn_scan_batch where gdn_scan_batch2 does not fit (MetalEnc.swift:760-777).
    if (dS != 128)
        return gd_gdn_scan_batch_serial(ctx, convOutN, keyDim, valueDim, convDim, gN, betaN, S,
                                        oN, nV, nK, dS, qScale, N);
    return gd_gdn_prefill(ctx, N, nV, nK, dS, dS, convOutN, convDim, convOutN + keyDim, convDim,
                          convOutN + 2 * keyDim, convDim, GD_F32, gN, betaN, S, oN, valueDim,
                          GD_F32, qScale, 64);
}
