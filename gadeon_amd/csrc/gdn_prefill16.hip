// Chunked (WY / UT) Gated DeltaNet prefill with f16 q, k, v: the algebra and
// symbols of gdn_prefill.hip (whose kernels serve f32 rows), reworked so that
// the serial chain over the chunks stays in one wave's registers.
//   gdn_prep16  (value head, chunk): K K^T and Q K^T on the matrix cores give
//               A and P; I + A is inverted in 16 x 16 blocks (diagonal blocks
//               by forward substitution, one wave each, then the block below,
//               all 256 threads); then W = T X and U = T Y (the UT transform)
//               on the matrix cores.  The chunks are independent.
//   gdn_scan16  (value head, 16 columns of S): walks the chunks in order.  One
//               wave is the serial chain: delta = U - W S, S <- e^{G_L} S +
//               K^T (e^{G_L-G} delta), everything it carries in its
//               registers; a second wave forms O = qScale (e^G (Q S) + P
//               delta) beside the next chunk.  Value columns of S are
//               independent, which is what splits the serial part across
//               workgroups.
// Operands that are f32 by nature (S, delta, T, beta e^G k, beta v, P) are
// split into hi + lo f16 pairs as there; q, k and v are used as they are.
// Chunks are of 32 tokens whichever chunk length the caller names: the sums
// are the same, and chunks of 64 were the slower at every shape measured (16
// heads, T = 512: 39 us against 30 before this; a 64 x 64 inverse has three
// more dependent block levels, and half the units).
// Workspace per (head, chunk) unit, every operand in the order in which the
// scan's lanes load it (one contiguous KiB per load instruction): W hi/lo,
// U, P hi/lo, e^G and e^{G_L-G}; per (key head, chunk) K^T.  Rows past a
// chunk's tokens are zero.
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
    float *G;         // [u][2][CP]: e^G, e^{G_L - G}
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

__global__ __launch_bounds__(256) void gdn_prep16(PrepArgs a) {
    __shared__ __attribute__((aligned(16))) f16 Ks[CP][PADK];
    __shared__ __attribute__((aligned(16))) f16 QVs[CP][PADK];     // Q, later V
    __shared__ __attribute__((aligned(16))) f16 Xh[DK][CP + 8], Xl[DK][CP + 8];
    __shared__ __attribute__((aligned(16))) f16 Yh[DV][CP + 8], Yl[DV][CP + 8];
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
    // K^T does not depend on the value head: the first of a key head writes it.
    const bool first = hv == hk;
    const int lr = lane & 15, kg = lane >> 4;

    // Rows of K and Q (and V, kept in registers until Q is done): thread e
    // handles 8 consecutive elements of row e / 16.
    // Every load goes out before any is converted (rows past the chunk read
    // token 0 and are zeroed at conversion): loads under a branch, converted
    // on arrival, waited for one by one.
    constexpr int NE = CP * DK / 8 / 256;                   // entries per thread
    u32x4 rk[NE], rq[NE], rv[NE];
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + 256 * n, t = e >> 4, i8 = (e & 15) * 8;
        const int64_t tok = t0 + (t < L ? t : 0);
        rk[n] = *(const u32x4 *)((const uint16_t *)a.k + tok * a.k_stride + (int64_t)hk * DK + i8);
        rq[n] = *(const u32x4 *)((const uint16_t *)a.q + tok * a.q_stride + (int64_t)hk * DK + i8);
        rv[n] = *(const u32x4 *)((const uint16_t *)a.v + tok * a.v_stride + (int64_t)hv * DV + i8);
    }
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + 256 * n, t = e >> 4, i8 = (e & 15) * 8;
        const u32x4 z = {0u, 0u, 0u, 0u};
        *(u32x4 *)&Ks[t][i8] = t < L ? rk[n] : z;
        *(u32x4 *)&QVs[t][i8] = t < L ? rq[n] : z;
        rv[n] = t < L ? rv[n] : z;
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
                acc = isP ? mfma(sv, tv, acc) : mfma(tv, sv, acc);
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
    // V replaces Q.
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + 256 * n, t = e >> 4, i8 = (e & 15) * 8;
        *(u32x4 *)&QVs[t][i8] = rv[n];
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
    for (int e = tid; e < DK * (CP / 8); e += 256) {
        const int g = e / DK, i = e % DK;
        float xv[8], yv[8];
        f16x8 kv;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int s = 8 * g + q;
            kv[q] = Ks[s][i];
            xv[q] = BEs[s] * (float)kv[q];
            yv[q] = Bs[s] * (float)QVs[s][i];
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
        if (first) *(f16x8 *)&a.w.KT[ki] = kv;
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
// waits for another wave: 40 MFMAs and the splits.  The
// output wave computes O = qScale (e^G (Q S) + P delta) of a chunk beside the
// chain's state update and next delta, from the split of S and delta that the
// chain leaves in LDS (by chunk parity: one barrier per chunk).
//   Operands come one contiguous KiB per load, refilled for the next chunk as
// soon as this one has used them.  (Two register sets, two chunks ahead, do
// not fit 256 registers: the accumulators then move through AGPRs, 23.5 us.)
//   16 heads, T = 512 (16 chunks): 15.6 us, 1 us a chunk (a chain of four
// waves that exchanged S and delta through LDS, two barriers a chunk: 22 at
// chunks of 64).  What bounds it is that chain of dependent MFMAs and splits.
constexpr int SCAN_THREADS = 128;     // chain wave, output wave

// The chain's operands of one chunk.
struct ChainRegs {
    f16x8 wh[2][4], wl[2][4];             // -W by token tile, key group
    f32x4 u[2], ed[2];                    // U and e^{G_L - G} of tokens 8g + 4m + v
    float dec;                            // e^{G_L}
    f16x8 ka[8];                          // K^T by key tile
};

// Eight f32 in two accumulators -> the operand fragment they make, split.
__device__ __forceinline__ void split_tiles(const f32x4 &x, const f32x4 &y, f16x8 &hi, f16x8 &lo) {
    const float f[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    split8(f, hi, lo);
}

template <typename OT>
__global__ __launch_bounds__(SCAN_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_scan16(ScanArgs a) {
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
        auto loadW = [&](int c, ChainRegs &k) {
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
        auto loadK = [&](int c, ChainRegs &k) {
            const size_t un = (size_t)hk * a.nchunks + min(c, a.nchunks - 1);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                k.ka[i] = *(const f16x8 *)(a.w.KT + un * KFRAG + (i * 64 + lane) * 8);
            }
        };
        auto chunk = [&](int c, ChainRegs &k) {
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
                    st[i] = acc;
                }
                split_tiles(st[2 * p], st[2 * p + 1], sh[p], sl_[p]);
            }
            __builtin_amdgcn_sched_barrier(0);
            loadK(c + 1, k);
            __builtin_amdgcn_sched_barrier(0);
        };
        ChainRegs k;
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
        // Q, P and e^G of tokens 16 m + lr: refilled for the next chunk as soon
        // as they are used.
        f16x8 qr[2][4], ph[2], pl[2];
        float eg[2];
        // Vector stores where every row keeps their alignment.
        const bool vec = ((uintptr_t)a.o % (4 * sizeof(OT))) == 0 && a.o_stride % 4 == 0;
        auto loadQ = [&](int c) {
            const int64_t t0 = (int64_t)min(c, a.nchunks - 1) * CP;
            const int L = (int)min((int64_t)CP, a.T - t0);
            // Rows past the chunk: its last token's (not stored).
#pragma unroll
            for (int m = 0; m < 2; m++)
#pragma unroll
                for (int p = 0; p < 4; p++)
                    qr[m][p] = *(const f16x8 *)((const uint16_t *)a.q + (t0 + min(16 * m + lr, L - 1)) * a.q_stride +
                                                (int64_t)hk * DK + 32 * p + 8 * g);
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
                    o[m] = mfma(sh, qr[m][p], o[m]);
                    o[m] = mfma(sl_, qr[m][p], o[m]);
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

}  // namespace

size_t gd_gdn_prefill16_bytes(int64_t T, int nV, int nK) {
    const size_t chunks = (size_t)((T + CP - 1) / CP), units = nV * chunks, kunits = std::min(nV, nK) * chunks;
    return units * (2 * WFRAG * 2 + UFRAG * 4 + 2 * PFRAG * 2 + 2 * CP * 4) + kunits * KFRAG * 2;
}

// Prep and scan with their per-(head, chunk) operands in ws (at least
// gd_gdn_prefill16_bytes).  Every byte of ws the scan reads is written by prep
// in the same call, so ws needs no clearing.
int gd_gdn_prefill16(gd_ctx *ctx, void *ws, int64_t T, int nV, int nK, const void *q, int64_t q_stride,
                     const void *k, int64_t k_stride, const void *v, int64_t v_stride, const float *g,
                     const float *beta, float *S, void *o, int64_t o_stride, int o_dtype, float qScale) {
    const int nchunks = (int)((T + CP - 1) / CP);
    const size_t units = (size_t)nV * nchunks, kunits = (size_t)std::min(nV, nK) * nchunks;
    uint8_t *p = (uint8_t *)ws;
    auto take = [&](size_t bytes) { uint8_t *r = p; p += bytes; return r; };
    Work w{};
    w.Wh = (f16 *)take(units * WFRAG * 2);
    w.Wl = (f16 *)take(units * WFRAG * 2);
    w.U = (float *)take(units * UFRAG * 4);
    w.Ph = (f16 *)take(units * PFRAG * 2);
    w.Pl = (f16 *)take(units * PFRAG * 2);
    w.KT = (f16 *)take(kunits * KFRAG * 2);
    w.G = (float *)take(units * 2 * CP * 4);
    const PrepArgs pa{q, k, v, q_stride, k_stride, v_stride, g, beta, w, T, nV, nK, nchunks};
    const ScanArgs sa{q, q_stride, w, S, o, o_stride, T, nV, nK, nchunks, qScale};
    hipLaunchKernelGGL(gdn_prep16, dim3((unsigned)units), dim3(256), 0, ctx->stream, pa);
    GD_LAUNCHED(ctx, "gdn_prep");
    const dim3 grid((unsigned)(nV * (DV / NCOL)));
    if (o_dtype == GD_F32)
        hipLaunchKernelGGL(gdn_scan16<float>, grid, dim3(SCAN_THREADS), 0, ctx->stream, sa);
    else
        hipLaunchKernelGGL(gdn_scan16<uint16_t>, grid, dim3(SCAN_THREADS), 0, ctx->stream, sa);
    GD_LAUNCHED(ctx, "gdn_scan");
    return GD_OK;
}
