// Gated DeltaNet glue and the per-token recurrence.
//
// Reference: GDN.step (LLM/src/SIMD/GDN.swift:20-120), the Metal kernels
// gdn_gate / gdn_conv / l2norm_rows / rmsnorm_rows / gdn_scan
// (LLM/metal/Kernels.metal:751-809, 1118-1243) and their MetalEnc hosts
// (LLM/src/Metal/MetalEnc.swift:213-272, 572-653).
//
// The fused decode step keeps one value column per lane: column j of the
// state, S[:, j], is all a lane needs (sk_j, delta_j, o_j are per-column), so
// a head's 64 KB state is read once and written once with no cross-lane
// reduction inside a wave; four waves split the key rows and meet once in LDS
// per reduction.  L2 normalization of q and k is folded into scalars:
// S^T k_hat = rk * S^T k and k_hat delta^T = k (rk * delta)^T.
#include "gd_internal.h"

// ------------------------------------------------------------------- gates

__global__ void gd_gate_kernel(const float *bPre, const float *aPre, const float *dt,
                               const float *aNeg, float *beta, float *g, int nV, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int h = (int)(i % nV);
    beta[i] = gd_sigmoid(bPre[i]);
    g[i] = gd_softplus(aPre[i] + dt[h]) * aNeg[h];
}

extern "C" int gd_gdn_gate(gd_ctx *ctx, const float *bPre, const float *aPre, const float *dt,
                           const float *aNeg, float *beta, float *g, int nV, int64_t count) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, bPre && aPre && dt && aNeg && beta && g, "gd_gdn_gate: null pointer");
    GD_REQUIRE(ctx, nV > 0 && count >= 0, "gd_gdn_gate: nV=%d count=%lld", nV, (long long)count);
    if (!count) return GD_OK;
    hipLaunchKernelGGL(gd_gate_kernel, dim3(gd_blocks(count, 256)), dim3(256), 0, ctx->stream,
                       bPre, aPre, dt, aNeg, beta, g, nV, count);
    GD_LAUNCHED(ctx, "gdn_gate");
    return GD_OK;
}

// ------------------------------------------------------------ causal conv

// One thread per channel; the ring stays in registers across the N tokens.
// window = [ring[0..dConv-2], x]; out = silu(sum window[j] * cw[c*dConv + j]).
// Serial over the tokens: every x of a channel is read before the outputs
// after it are written, so out may overlap x (the tiled kernel below may not).
template <int KC>
__global__ void gd_conv_kernel(const float *x, float *ring, const float *cw, float *out,
                               int convDim, int64_t N) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= convDim) return;
    float w[KC], r[KC];
#pragma unroll
    for (int j = 0; j < KC; j++) w[j] = cw[(int64_t)c * KC + j];
#pragma unroll
    for (int j = 0; j + 1 < KC; j++) r[j] = ring[(int64_t)j * convDim + c];
    for (int64_t n = 0; n < N; n++) {
        const float cur = x[n * convDim + c];
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j + 1 < KC; j++) acc += r[j] * w[j];
        acc += cur * w[KC - 1];
        out[n * convDim + c] = gd_silu(acc);
#pragma unroll
        for (int j = 0; j + 2 < KC; j++) r[j] = r[j + 1];
        if (KC >= 2) r[KC - 2] = cur;
    }
#pragma unroll
    for (int j = 0; j + 1 < KC; j++) ring[(int64_t)j * convDim + c] = r[j];
}

// V consecutive floats.
template <int V> struct Floats { float v[V]; };
template <int V> __device__ __forceinline__ Floats<V> ld_floats(const float *p) {
    Floats<V> r;
    if constexpr (V == 4) {
        const f32x4 a = *(const f32x4 *)p;
#pragma unroll
        for (int i = 0; i < 4; i++) r.v[i] = a[i];
    } else {
        r.v[0] = *p;
    }
    return r;
}
template <int V> __device__ __forceinline__ void st_floats(float *p, const Floats<V> &r) {
    if constexpr (V == 4) *(f32x4 *)p = f32x4{r.v[0], r.v[1], r.v[2], r.v[3]};
    else *p = r.v[0];
}

// The same conv with the tokens in tiles of TT: a thread holds V channels and
// slides its window over the tile, its TT + KC - 1 input rows all requested
// before the first is used.  Memory-bound (x read and out written once, plus
// the KC - 1 rows a tile reads of the one before it): 1000 tokens x 10240
// channels 327 us with one thread per channel walking all tokens (40
// workgroups, one load in flight each), 20 us here (4.1 TB/s of x and out; a
// large copy runs at 4.7).  Only tile 0 reads the ring
// (TT >= KC - 1), so it alone advances it, after its reads, to the last KC - 1
// inputs (N >= KC - 1: fewer tokens take the serial kernel).
template <int KC, int V, int TT>
__global__ __launch_bounds__(256) void gd_conv_tile_kernel(const float *__restrict__ x, float *ring,
                                                           const float *__restrict__ cw,
                                                           float *__restrict__ out, int convDim,
                                                           int64_t N) {
    static_assert(TT >= KC - 1, "only tile 0 may reach back into the ring");
    const int c = (blockIdx.x * 256 + threadIdx.x) * V;
    if (c >= convDim) return;
    const int64_t n0 = (int64_t)blockIdx.y * TT;
    Floats<V> win[TT + KC - 1];                          // win[j]: token n0 - (KC - 1) + j
    float w[V][KC];
#pragma unroll
    for (int j = 0; j < TT + KC - 1; j++) {
        const int64_t m = n0 - (KC - 1) + j;
        win[j] = ld_floats<V>(x + (m < 0 ? 0 : m < N ? m : N - 1) * convDim + c);
    }
#pragma unroll
    for (int i = 0; i < V; i++)
#pragma unroll
        for (int j = 0; j < KC; j++) w[i][j] = cw[(int64_t)(c + i) * KC + j];
    if (n0 == 0) {
#pragma unroll
        for (int j = 0; j + 1 < KC; j++) win[j] = ld_floats<V>(ring + (int64_t)j * convDim + c);
    }
#pragma unroll
    for (int t = 0; t < TT; t++) {
        if (n0 + t >= N) break;
        Floats<V> y;
#pragma unroll
        for (int i = 0; i < V; i++) {
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < KC; j++) acc += win[t + j].v[i] * w[i][j];
            y.v[i] = gd_silu(acc);
        }
        st_floats<V>(out + (n0 + t) * convDim + c, y);
    }
    if (n0 == 0) {
#pragma unroll
        for (int j = 0; j + 1 < KC; j++)
            st_floats<V>(ring + (int64_t)j * convDim + c, ld_floats<V>(x + (N - (KC - 1) + j) * convDim + c));
    }
}

// The tiled conv where nothing the tiles write is read by another tile: out
// and ring apart from each other and from the inputs.  Four channels a thread
// where rows keep 16-byte alignment.  Tiles of 16 tokens (a fifth more rows
// read than the input has) once they fill the chip twice over, else of 4 (8
// where the window is longer), so that short inputs spread over more CUs.
//   Up to 10 tokens walk the channels: 1.8 us and 0.2 a token for a chain of
// calls, at 4096 to 10240 channels alike, where the tiles, a quarter of the
// workgroups and a window of loads each, take 2.9 (one token) to 3.7 (from 4
// on): 1, 4, 8 and 12 tokens 2.0, 2.4, 3.2 and 4.1 us (tiles 2.9, 3.7, 3.7, 3.7).
constexpr int CONV_SERIAL = 10;
template <int KC>
static bool launch_conv_tiles(gd_ctx *ctx, const float *x, float *ring, const float *cw, float *out,
                              int convDim, int64_t N) {
    static_assert(CONV_SERIAL >= KC - 1, "the tiles advance the ring from x alone");
    if (N <= CONV_SERIAL) return false;
    auto apart = [](const void *a, size_t an, const void *b, size_t bn) {
        const uintptr_t p = (uintptr_t)a, q = (uintptr_t)b;
        return p + an <= q || q + bn <= p;
    };
    const size_t xb = (size_t)N * convDim * 4, rb = (size_t)(KC - 1) * convDim * 4, wb = (size_t)convDim * KC * 4;
    if (!apart(x, xb, out, xb) || !apart(cw, wb, out, xb)) return false;
    if (KC > 1 && !(apart(ring, rb, out, xb) && apart(ring, rb, x, xb) && apart(ring, rb, cw, wb)))
        return false;
    constexpr int TS = KC <= 5 ? 4 : 8, TL = 16;
    const bool vec = convDim % 4 == 0 &&
                     (((uintptr_t)x | (uintptr_t)out | (KC > 1 ? (uintptr_t)ring : 0)) & 15) == 0;
    const unsigned gx = gd_blocks(convDim, vec ? 1024 : 256);
    const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    const bool large = (int64_t)gx * ((N + TL - 1) / TL) >= 2 * cus;
    const int64_t gy = (N + (large ? TL : TS) - 1) / (large ? TL : TS);
    if (gy > 65535) return false;
    const dim3 g(gx, (unsigned)gy), b(256);
#define GD_CONV_TILE(V_, T_) hipLaunchKernelGGL((gd_conv_tile_kernel<KC, V_, T_>), g, b, 0, ctx->stream, \
                                                x, ring, cw, out, convDim, N)
    if (vec) { if (large) GD_CONV_TILE(4, TL); else GD_CONV_TILE(4, TS); }
    else { if (large) GD_CONV_TILE(1, TL); else GD_CONV_TILE(1, TS); }
#undef GD_CONV_TILE
    return true;
}

extern "C" int gd_gdn_conv(gd_ctx *ctx, const float *qkvMix, float *convState, const float *cw,
                           float *out, int convDim, int dConv, int64_t N) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, qkvMix && cw && out && (convState || dConv == 1), "gd_gdn_conv: null pointer");
    GD_REQUIRE(ctx, convDim > 0 && N >= 0, "gd_gdn_conv: convDim=%d N=%lld", convDim, (long long)N);
    GD_REQUIRE(ctx, dConv >= 1 && dConv <= 8, "gd_gdn_conv: dConv=%d not in [1,8]", dConv);
    if (!N) return GD_OK;
    dim3 g(gd_blocks(convDim, 256)), b(256);
    switch (dConv) {
#define GD_CONV_CASE(KC) \
    case KC: if (!launch_conv_tiles<KC>(ctx, qkvMix, convState, cw, out, convDim, N)) \
            hipLaunchKernelGGL(gd_conv_kernel<KC>, g, b, 0, ctx->stream, qkvMix, convState, cw, \
                               out, convDim, N); break;
        GD_CONV_CASE(1) GD_CONV_CASE(2) GD_CONV_CASE(3) GD_CONV_CASE(4)
        GD_CONV_CASE(5) GD_CONV_CASE(6) GD_CONV_CASE(7) GD_CONV_CASE(8)
#undef GD_CONV_CASE
    }
    GD_LAUNCHED(ctx, "gdn_conv");
    return GD_OK;
}

// ------------------------------------------------------------------- norms

// One 64-lane wave per row.
__global__ void gd_l2norm_kernel(float *x, int d, int rowsPerTok, int64_t tokStride,
                                 int64_t rows, float eps) {
    const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    float *r = x + (row / rowsPerTok) * tokStride + (row % rowsPerTok) * d;
    float ss = 0.0f;
    for (int i = lane; i < d; i += 64) ss += r[i] * r[i];
    ss = gd_wave_sum(ss);
    const float s = 1.0f / sqrtf(ss + eps);
    for (int i = lane; i < d; i += 64) r[i] *= s;
}

extern "C" int gd_l2norm_rows(gd_ctx *ctx, float *x, int d, int rowsPerTok, int64_t tokStride,
                              int64_t tokens, float eps) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, x && d > 0 && rowsPerTok > 0 && tokens >= 0 &&
                        tokStride >= (int64_t)rowsPerTok * d,
               "gd_l2norm_rows: bad arguments");
    const int64_t rows = (int64_t)rowsPerTok * tokens;
    if (!rows) return GD_OK;
    hipLaunchKernelGGL(gd_l2norm_kernel, dim3(gd_blocks(rows, 4)), dim3(256), 0, ctx->stream, x,
                       d, rowsPerTok, tokStride, rows, eps);
    GD_LAUNCHED(ctx, "l2norm_rows");
    return GD_OK;
}

__global__ void gd_rmsnorm_rows_kernel(float *x, int d, int64_t rows, const float *w, float eps) {
    const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    float *r = x + row * d;
    float ss = 0.0f;
    for (int i = lane; i < d; i += 64) ss += r[i] * r[i];
    ss = gd_wave_sum(ss);
    const float s = 1.0f / sqrtf(ss / (float)d + eps);
    for (int i = lane; i < d; i += 64) r[i] = r[i] * s * w[i];
}

// Rows of 4 L elements, a row in L lanes' registers (16 bytes a lane) and four
// rows a thread in flight.  Bound by HBM: 48000 rows of 128 (49 MB) 8.7 us,
// one row a wave and 4 bytes a lane 13.8.
template <int L>
__global__ __launch_bounds__(256) void gd_rmsnorm_rows_vec_kernel(float *x, int64_t rows, const float *w, float eps) {
    constexpr int NR = 4, D = 4 * L, G = 256 / L;
    const int l = threadIdx.x % L;
    const int64_t r0 = (int64_t)blockIdx.x * (G * NR) + threadIdx.x / L;
    const f32x4 wv = *(const f32x4 *)(w + 4 * l);
    f32x4 v[NR];
#pragma unroll
    for (int k = 0; k < NR; k++) v[k] = *(const f32x4 *)(x + min(r0 + G * k, rows - 1) * D + 4 * l);
#pragma unroll
    for (int k = 0; k < NR; k++) {
        float ss = (v[k][0] * v[k][0] + v[k][1] * v[k][1]) + (v[k][2] * v[k][2] + v[k][3] * v[k][3]);
#pragma unroll
        for (int o = L / 2; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
        const float s = 1.0f / sqrtf(ss / (float)D + eps);
        if (r0 + G * k < rows) *(f32x4 *)(x + (r0 + G * k) * D + 4 * l) = v[k] * s * wv;
    }
}

extern "C" int gd_rmsnorm_rows(gd_ctx *ctx, float *x, int d, int64_t rows, const float *w,
                               float eps) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, x && w && d > 0 && rows >= 0, "gd_rmsnorm_rows: bad arguments");
    if (!rows) return GD_OK;
    // The head dims of the models, 16-byte rows, from 2^20 elements on: fewer
    // leave CUs without a block of 32 (16) rows and pay for its longer chain.  A
    // chain of calls, rows of 128: 1000 2.2 us (vector kernel 2.8), 6000 3.1
    // (3.2), 8000 3.4 (3.3), 16000 5.0 (3.9), 48000 13.8 (8.8); rows of 256: 1000
    // 2.7 (3.0), 4000 3.4 (3.4), 8000 4.5 (4.1).
    const bool al = (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && rows * d >= 1 << 20;
    if (d == 128 && al)
        hipLaunchKernelGGL(gd_rmsnorm_rows_vec_kernel<32>, dim3(gd_blocks(rows, 32)), dim3(256), 0, ctx->stream, x,
                           rows, w, eps);
    else if (d == 256 && al)
        hipLaunchKernelGGL(gd_rmsnorm_rows_vec_kernel<64>, dim3(gd_blocks(rows, 16)), dim3(256), 0, ctx->stream, x,
                           rows, w, eps);
    else
        hipLaunchKernelGGL(gd_rmsnorm_rows_kernel, dim3(gd_blocks(rows, 4)), dim3(256), 0,
                           ctx->stream, x, d, rows, w, eps);
    GD_LAUNCHED(ctx, "rmsnorm_rows");
    return GD_OK;
}

// The row held in the registers of NT threads, NP 16-byte pieces each: a row is
// read once, with its weights requested beside it.  Bound by two latencies of
// memory and the block's sum; one float a lane in a loop, read twice, took 11.6
// us for 27 as for 333 rows of 5120, this (512 x 4) 2.5 and 4.5.
template <int YT, int NT, int NP>
__global__ __launch_bounds__(NT) void gd_rmsnorm_vec_kernel(const float *x, const float *w, void *y, int n,
                                                            float eps) {
    __shared__ float red[NT / 64];
    const int64_t row = blockIdx.x;
    const float *xr = x + row * n;
    f32x4 v[NP], ww[NP];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NP; k++) {
        const int i = 4 * (threadIdx.x + NT * k);
        if (i >= n) break;
        v[k] = *(const f32x4 *)(xr + i);
        ww[k] = *(const f32x4 *)(w + i);
    }
#pragma unroll
    for (int k = 0; k < NP; k++) {
        if (4 * ((int)threadIdx.x + NT * k) >= n) break;
        ss += (v[k][0] * v[k][0] + v[k][1] * v[k][1]) + (v[k][2] * v[k][2] + v[k][3] * v[k][3]);
    }
    ss = gd_block_sum(ss, red);
    const float s = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
    for (int k = 0; k < NP; k++) {
        const int i = 4 * (threadIdx.x + NT * k);
        if (i >= n) break;
        const f32x4 o = v[k] * s * ww[k];
        if (YT == GD_F32) {
            *(f32x4 *)((float *)y + row * n + i) = o;
        } else {
            const uint32_t lo = (uint32_t)gd_f2h(o[0]) | ((uint32_t)gd_f2h(o[1]) << 16);
            const uint32_t hi = (uint32_t)gd_f2h(o[2]) | ((uint32_t)gd_f2h(o[3]) << 16);
            *(u32x2 *)((uint16_t *)y + row * n + i) = u32x2{lo, hi};
        }
    }
}

// One 256-thread block per row of length n, any n and alignment.
template <int YT>
__global__ void gd_rmsnorm_kernel(const float *x, const float *w, void *y, int64_t n, float eps) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const float *xr = x + row * n;
    float ss = 0.0f;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) ss += xr[i] * xr[i];
    ss = gd_block_sum(ss, red);
    const float s = 1.0f / sqrtf(ss / (float)n + eps);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const float v = xr[i] * s * w[i];
        if (YT == GD_F32) ((float *)y)[row * n + i] = v;
        else ((uint16_t *)y)[row * n + i] = gd_f2h(v);
    }
}

extern "C" int gd_rmsnorm(gd_ctx *ctx, const float *x, const float *w, void *y, int y_dtype,
                          int64_t n, int64_t rows, float eps) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, x && w && y && n > 0 && rows >= 0, "gd_rmsnorm: bad arguments");
    GD_REQUIRE(ctx, y_dtype == GD_F32 || y_dtype == GD_F16, "gd_rmsnorm: bad dtype");
    GD_REQUIRE(ctx, rows < (1LL << 31), "gd_rmsnorm: too many rows");
    if (!rows) return GD_OK;
    // Rows of whole 16-byte pieces that fit the registers (27 rows of 5120: 2.5
    // us, a float a lane 11.6), in 512 threads, or in 128 where those hold the
    // row.  A launch holds fewer than 2^32 threads: rows past that go a float a lane.
    const int nt = n <= 512 ? 128 : 512;
    const bool vec = n % 4 == 0 && n <= 8192 && (uint64_t)rows * nt < (1ULL << 32) &&
                     (((uintptr_t)x | (uintptr_t)w) & 15) == 0 &&
                     ((uintptr_t)y & (y_dtype == GD_F32 ? 15 : 7)) == 0;
#define GD_RMS(K_, NT_, N_) hipLaunchKernelGGL(K_, dim3((unsigned)rows), dim3(NT_), 0, ctx->stream, x, w, y, N_, eps)
    if (vec && nt == 128) {
        if (y_dtype == GD_F32) GD_RMS((gd_rmsnorm_vec_kernel<GD_F32, 128, 1>), 128, (int)n);
        else GD_RMS((gd_rmsnorm_vec_kernel<GD_F16, 128, 1>), 128, (int)n);
    } else if (vec) {
        if (y_dtype == GD_F32) GD_RMS((gd_rmsnorm_vec_kernel<GD_F32, 512, 4>), 512, (int)n);
        else GD_RMS((gd_rmsnorm_vec_kernel<GD_F16, 512, 4>), 512, (int)n);
    } else {
        if (y_dtype == GD_F32) GD_RMS(gd_rmsnorm_kernel<GD_F32>, 256, n);
        else GD_RMS(gd_rmsnorm_kernel<GD_F16>, 256, n);
    }
#undef GD_RMS
    GD_LAUNCHED(ctx, "rmsnorm");
    return GD_OK;
}

// ------------------------------------------------------------- elementwise

template <int OP>
__global__ void gd_elementwise_kernel(float *a, const float *b, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (OP == 0) a[i] = gd_silu(a[i]) * b[i];
    else if (OP == 1) a[i] = a[i] * gd_silu(b[i]);
    else a[i] += b[i];
}

template <int OP>
static int elementwise(gd_ctx *ctx, float *a, const float *b, int64_t n, const char *name) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, a && b && n >= 0, "%s: bad arguments", name);
    if (!n) return GD_OK;
    hipLaunchKernelGGL(gd_elementwise_kernel<OP>, dim3(gd_blocks(n, 256)), dim3(256), 0,
                       ctx->stream, a, b, n);
    GD_LAUNCHED(ctx, name);
    return GD_OK;
}

extern "C" int gd_silu_mul(gd_ctx *ctx, float *a, const float *b, int64_t n) {
    return elementwise<0>(ctx, a, b, n, "silu_mul");
}
extern "C" int gd_mul_silu(gd_ctx *ctx, float *a, const float *b, int64_t n) {
    return elementwise<1>(ctx, a, b, n, "mul_silu");
}
extern "C" int gd_add(gd_ctx *ctx, float *x, const float *y, int64_t n) {
    return elementwise<2>(ctx, x, y, n, "add_inplace");
}

// -------------------------------------------------- fused state-carry decode

namespace {

constexpr int DEC_DS = 128;      // state size handled by the fused kernel
constexpr int DEC_COLS = 64;     // value columns per workgroup (one per lane)
constexpr int DEC_ROWS = 32;     // key rows per wave (4 waves)

template <typename T> __device__ __forceinline__ float ld(const T *p, int64_t i);
template <> __device__ __forceinline__ float ld<float>(const float *p, int64_t i) { return p[i]; }
template <> __device__ __forceinline__ float ld<uint16_t>(const uint16_t *p, int64_t i) {
    return gd_h2f(p[i]);
}
template <typename T> __device__ __forceinline__ void st(T *p, int64_t i, float v);
template <> __device__ __forceinline__ void st<float>(float *p, int64_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void st<uint16_t>(uint16_t *p, int64_t i, float v) {
    p[i] = gd_f2h(v);
}

// Grid: (dS/64 column blocks, nV heads, B sequences); 256 threads.
// NORM: L2-normalize q,k.  GATE: beta/g from pre-activations with dt/aNeg.
template <typename IO, bool NORM, bool GATE>
__global__ __launch_bounds__(256) void gd_decode_kernel(
        const IO *__restrict__ q, const IO *__restrict__ k, const IO *__restrict__ v,
        const float *__restrict__ g_in, const float *__restrict__ beta_in,
        const float *__restrict__ dt, const float *__restrict__ aNeg, float *__restrict__ S,
        IO *__restrict__ o, int nV, int nK, float qScale, float eps) {
    __shared__ float kq[2][DEC_DS];
    __shared__ float red[4][DEC_COLS];
    __shared__ float scal[2];

    const int jb = blockIdx.x, hv = blockIdx.y, b = blockIdx.z;
    const int hk = hv % nK;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = jb * DEC_COLS + lane;

    const int64_t qk_off = ((int64_t)b * nK + hk) * DEC_DS;
    const int64_t v_off = ((int64_t)b * nV + hv) * DEC_DS;
    const int64_t gb = (int64_t)b * nV + hv;
    float *Sh = S + ((int64_t)b * nV + hv) * DEC_DS * DEC_DS;

    // Issue the state loads first: they are the bandwidth.
    float s[DEC_ROWS];
#pragma unroll
    for (int r = 0; r < DEC_ROWS; r++) s[r] = Sh[(int64_t)(wave * DEC_ROWS + r) * DEC_DS + j];

    if (tid < DEC_DS) kq[0][tid] = ld(k, qk_off + tid);
    else kq[1][tid - DEC_DS] = ld(q, qk_off + tid - DEC_DS);
    float beta, gam;
    if (GATE) {
        beta = gd_sigmoid(beta_in[gb]);
        gam = expf(gd_softplus(g_in[gb] + dt[hv]) * aNeg[hv]);
    } else {
        beta = beta_in[gb];
        gam = expf(g_in[gb]);
    }
    const float vj = ld(v, v_off + j);
    __syncthreads();
    float rk = 1.0f, rq = 1.0f;
    if (NORM) {
        // Waves 0/1 reduce |k|^2 and |q|^2 (2 elements per lane).
        if (wave < 2) {
            const float a = kq[wave][lane], c = kq[wave][lane + 64];
            const float ss = gd_wave_sum(a * a + c * c);
            if (lane == 0) scal[wave] = 1.0f / sqrtf(ss + eps);
        }
        __syncthreads();
        rk = scal[0];
        rq = scal[1];
    }

    // Decay and this wave's part of S^T k.
    float sk = 0.0f;
#pragma unroll
    for (int r = 0; r < DEC_ROWS; r++) {
        s[r] *= gam;
        sk = fmaf(s[r], kq[0][wave * DEC_ROWS + r], sk);
    }
    red[wave][lane] = sk;
    __syncthreads();
    sk = (red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane]) * rk;
    const float delta = beta * (vj - sk) * rk;   // rk folds k_hat into the update
    __syncthreads();                              // red[] is reused below

    float acc = 0.0f;
#pragma unroll
    for (int r = 0; r < DEC_ROWS; r++) {
        const int i = wave * DEC_ROWS + r;
        s[r] = fmaf(kq[0][i], delta, s[r]);
        acc = fmaf(s[r], kq[1][i], acc);
        Sh[(int64_t)i * DEC_DS + j] = s[r];
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
        const float oj = (red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane]) * rq * qScale;
        st(o, v_off + j, oj);
    }
}

// General-dS single-token scan for shapes the fused kernel does not take: one
// thread per (value head, column), as gdn_scan (Kernels.metal:1206-1243).
__global__ void gd_scan_generic_kernel(const float *q, const float *k, const float *v,
                                       const float *g, const float *beta, float *S, float *o,
                                       int nV, int nK, int dS, float qScale) {
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= nV * dS) return;
    const int hv = gid / dS, j = gid % dS, hk = hv % nK;
    const float *qh = q + (int64_t)hk * dS, *kh = k + (int64_t)hk * dS;
    float *Sh = S + (int64_t)hv * dS * dS;
    const float gam = expf(g[hv]), b = beta[hv];
    float sk = 0.0f;
    for (int i = 0; i < dS; i++) {
        const float x = Sh[(int64_t)i * dS + j] * gam;
        Sh[(int64_t)i * dS + j] = x;
        sk += x * kh[i];
    }
    const float d = b * (v[(int64_t)hv * dS + j] - sk);
    float acc = 0.0f;
    for (int i = 0; i < dS; i++) {
        const float x = Sh[(int64_t)i * dS + j] + kh[i] * d;
        Sh[(int64_t)i * dS + j] = x;
        acc += x * qh[i];
    }
    o[(int64_t)hv * dS + j] = acc * qScale;
}

// N tokens of the scan for state sizes the chunked prefill does not take
// (dS != 128): gdn_scan_batch (Kernels.metal:1525-1565), which
// MetalEnc.gdnScanBatch dispatches for any dS (MetalEnc.swift:741-778).  One
// workgroup per value head, thread j owning value column j of S (dS <= 1024),
// tokens in order; q and k of the token are staged once per workgroup in
// LDS (the column walks read them at every row), S stays in device memory
// as in the reference (a head's dS x dS f32 exceeds LDS beyond 181).
__global__ __launch_bounds__(1024) void gd_scan_batch_serial_kernel(
        const float *convOutN, const float *gN, const float *betaN, float *S, float *oN, int nV,
        int nK, int dS, float qScale, int64_t N, int convDim, int keyDim, int valueDim) {
    extern __shared__ float qk[];                 // [2][dS]: q, k of the token
    const int hv = blockIdx.x, j = threadIdx.x, hk = hv % nK;
    float *Sh = S + (int64_t)hv * dS * dS;
    for (int64_t n = 0; n < N; n++) {
        const float *row = convOutN + n * convDim;
        __syncthreads();                          // the previous token's reads are done
        for (int i = threadIdx.x; i < dS; i += blockDim.x) {
            qk[i] = row[(int64_t)hk * dS + i];
            qk[dS + i] = row[keyDim + (int64_t)hk * dS + i];
        }
        __syncthreads();
        if (j >= dS) continue;
        const float gam = expf(gN[n * nV + hv]), b = betaN[n * nV + hv];
        const float *k = qk + dS, *q = qk;
        float sk = 0.0f;
        for (int i = 0; i < dS; i++) {
            const float x = Sh[(int64_t)i * dS + j] * gam;
            Sh[(int64_t)i * dS + j] = x;
            sk += x * k[i];
        }
        const float d = b * (row[2 * (int64_t)keyDim + (int64_t)hv * dS + j] - sk);
        float acc = 0.0f;
        for (int i = 0; i < dS; i++) {
            const float x = Sh[(int64_t)i * dS + j] + k[i] * d;
            Sh[(int64_t)i * dS + j] = x;
            acc += x * q[i];
        }
        oN[n * valueDim + (int64_t)hv * dS + j] = acc * qScale;
    }
}

}  // namespace

// Token-serial gdnScanBatch for any dS up to 1024 (the caller has checked
// the pointers and the dimensions).
int gd_gdn_scan_batch_serial(gd_ctx *ctx, const float *convOutN, int keyDim, int valueDim,
                             int convDim, const float *gN, const float *betaN, float *S,
                             float *oN, int nV, int nK, int dS, float qScale, int64_t N) {
    GD_REQUIRE(ctx, dS > 0 && dS <= 1024 && nV > 0 && nK > 0 && nV <= 65535,
               "gd_gdn_scan_batch: dS=%d nV=%d nK=%d (the token-serial scan takes dS <= 1024)",
               dS, nV, nK);
    if (N <= 0) return GD_OK;
    const int threads = (dS + 63) / 64 * 64;
    hipLaunchKernelGGL(gd_scan_batch_serial_kernel, dim3(nV), dim3(threads),
                       (size_t)2 * dS * sizeof(float), ctx->stream, convOutN, gN, betaN, S, oN,
                       nV, nK, dS, qScale, N, convDim, keyDim, valueDim);
    GD_LAUNCHED(ctx, "gdn_scan_batch");
    return GD_OK;
}

extern "C" int gd_gdn_decode(gd_ctx *ctx, int B, int nV, int nK, int dS, const void *q,
                             const void *k, const void *v, int io_dtype, const float *g_in,
                             const float *beta_in, const float *dt, const float *aNeg, float *S,
                             void *o, float qScale, float eps) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, q && k && v && g_in && beta_in && S && o, "gd_gdn_decode: null pointer");
    GD_REQUIRE(ctx, (dt == nullptr) == (aNeg == nullptr),
               "gd_gdn_decode: dt and aNeg must both be given or both be NULL");
    GD_REQUIRE(ctx, B > 0 && nV > 0 && nK > 0 && B <= 65535 && nV <= 65535,
               "gd_gdn_decode: B=%d nV=%d nK=%d", B, nV, nK);
    GD_REQUIRE(ctx, dS == DEC_DS, "gd_gdn_decode: dS=%d (the fused step takes 128)", dS);
    GD_REQUIRE(ctx, io_dtype == GD_F32 || io_dtype == GD_F16, "gd_gdn_decode: bad dtype");
    dim3 grid(DEC_DS / DEC_COLS, nV, B), blk(256);
    const bool gate = dt != nullptr;
#define GD_DEC(IO, G) \
    hipLaunchKernelGGL((gd_decode_kernel<IO, true, G>), grid, blk, 0, ctx->stream, \
                       (const IO *)q, (const IO *)k, (const IO *)v, g_in, beta_in, dt, aNeg, S, \
                       (IO *)o, nV, nK, qScale, eps)
    if (io_dtype == GD_F32) { if (gate) GD_DEC(float, true); else GD_DEC(float, false); }
    else { if (gate) GD_DEC(uint16_t, true); else GD_DEC(uint16_t, false); }
#undef GD_DEC
    GD_LAUNCHED(ctx, "gdn_decode");
    return GD_OK;
}

extern "C" int gd_gdn_scan(gd_ctx *ctx, const float *q, const float *k, const float *v,
                           const float *g, const float *beta, float *S, float *o, int nV, int nK,
                           int dS, float qScale) {
    GD_CHECK_CTX(ctx);
    GD_REQUIRE(ctx, q && k && v && g && beta && S && o, "gd_gdn_scan: null pointer");
    GD_REQUIRE(ctx, nV > 0 && nK > 0 && dS > 0, "gd_gdn_scan: nV=%d nK=%d dS=%d", nV, nK, dS);
    if (dS == DEC_DS && nV <= 65535) {
        dim3 grid(DEC_DS / DEC_COLS, nV, 1);
        hipLaunchKernelGGL((gd_decode_kernel<float, false, false>), grid, dim3(256), 0,
                           ctx->stream, q, k, v, g, beta, nullptr, nullptr, S, o, nV, nK, qScale,
                           0.0f);
    } else {
        hipLaunchKernelGGL(gd_scan_generic_kernel, dim3(gd_blocks((int64_t)nV * dS, 256)),
                           dim3(256), 0, ctx->stream, q, k, v, g, beta, S, o, nV, nK, dS, qScale);
    }
    GD_LAUNCHED(ctx, "gdn_scan");
    return GD_OK;
}
