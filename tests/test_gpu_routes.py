"""The rules that send a call to one of two kernels, by time: where an entry
has a second kernel that a call can be put on (an output over its input, a
start off 16-byte alignment, a forced plan), the one that the rule picks for
the plain call is not the slower one.  Each side is a recorded chain of calls,
the fastest of several replays; 1.15 leaves room for the placement of buffers
and for the other kernel's own small costs, and the rules that these tests
were written against were off by 1.2 to 4."""
import ctypes as C

import numpy as np
import pytest

import gadeon_amd as ga

pytestmark = pytest.mark.gpu

EPS = 1e-6
SLACK = 1.15


def chain_ms(ctx, call, n=50, replays=12):
    """Fastest replay of n recorded calls, after one direct call (workspaces)."""
    call()
    ctx.gd_graph_begin()
    for _ in range(n):
        call()
    g, ms, best = C.c_void_p(), C.c_float(), 1e9
    ctx.gd_graph_end(C.byref(g))
    for _ in range(replays):
        ctx.gd_timer_start()
        ctx.gd_graph_launch(g)
        ctx.gd_timer_stop(C.byref(ms))
        best = min(best, ms.value)
    ctx.lib.gd_graph_destroy(g)
    return best


def not_slower(ctx, picked, other, n=50):
    """Chains of the two calls, measured again where something else ran beside one."""
    for _ in range(3):
        a, b = chain_ms(ctx, picked, n), chain_ms(ctx, other, n)
        if a < SLACK * b:
            return
    assert a < SLACK * b


def zeros(ctx, nbytes):
    p = ctx.alloc(nbytes)
    ctx.gd_fill_u32(p, 0, nbytes // 4)
    return p


@pytest.mark.parametrize("N", [1, 4, 8, 10])
def test_conv_few_tokens(ctx, N):
    """Few tokens against the token-serial kernel, which a call takes whose
    output replaces its input."""
    cd = 8192
    x, o, ring, cw = (zeros(ctx, n * cd * 4) for n in (N, N, 3, 4))
    conv = lambda out: ctx.gd_gdn_conv(x, ring, cw, out, cd, 4, N)
    not_slower(ctx, lambda: conv(o), lambda: conv(x))
    for p in (x, o, ring, cw):
        ctx.free(p)


@pytest.mark.parametrize("d,rows", [(128, 64), (128, 1000), (256, 64), (128, 48000)])
def test_rmsnorm_rows_few(ctx, d, rows):
    """Few rows, and many, against the kernel for any alignment (w one float off)."""
    x, w = zeros(ctx, rows * d * 4), zeros(ctx, d * 4 + 16)
    norm = lambda weights: ctx.gd_rmsnorm_rows(x, d, rows, weights, EPS)
    not_slower(ctx, lambda: norm(w), lambda: norm(w + 4))
    for p in (x, w):
        ctx.free(p)


@pytest.mark.parametrize("n,rows", [(64, 20000), (128, 4000), (512, 20000), (1024, 20000)])
def test_rmsnorm_short_rows(ctx, n, rows):
    """Many short rows against the kernel for any alignment (w one float off)."""
    x, w, y = zeros(ctx, rows * n * 4), zeros(ctx, n * 4 + 16), zeros(ctx, rows * n * 4)
    norm = lambda weights: ctx.gd_rmsnorm(x, weights, y, ga.F32, n, rows, EPS)
    not_slower(ctx, lambda: norm(w), lambda: norm(w + 4), 20)
    for p in (x, w, y):
        ctx.free(p)


def test_rmsnorm_many_rows(ctx):
    """2^23 rows of 516: 512 threads a row are more than one launch holds."""
    n, rows = 516, 1 << 23
    x, w = ctx.alloc(rows * n * 4), ctx.put(np.ones(n, np.float32))
    ctx.gd_fill_u32(x, int(np.float32(3).view(np.uint32)), rows * n)
    ctx.gd_rmsnorm(x, w, x, ga.F32, n, rows, EPS)
    for r in (0, rows // 2, rows - 1):
        assert np.allclose(ctx.get(x + r * n * 4, n, np.float32), 1, rtol=1e-6)
    for p in (x, w):
        ctx.free(p)


@pytest.mark.parametrize("hd,nh,nkv,T", [(256, 8, 8, 1153), (256, 8, 8, 3000), (128, 16, 8, 577), (128, 16, 16, 640),
                                         (256, 24, 4, 9000), (256, 16, 16, 3000)])
def test_decode_attention_keys(ctx, hd, nh, nkv, T):
    """Few heads, or one a kv head, over middling contexts, and the usual long
    one, against the wave-a-key kernel, which a q off 16-byte alignment takes."""
    page, kv_dim = 16, nkv * hd
    npages = -(-T // page)
    kc, vc = (zeros(ctx, npages * page * kv_dim * 2) for _ in range(2))
    table = ctx.put(np.arange(npages, dtype=np.int32))
    q, gate, out, part = (zeros(ctx, n * 4 + 16) for n in (nh * hd, nh * hd, nh * hd, nh * 16 * (hd + 2)))
    call = lambda x: ctx.gd_attn_paged(x, kc, vc, table, gate, out, part, hd, nh, nkv, T, kv_dim, page,
                                       C.c_float(hd ** -0.5), 1, 0)
    not_slower(ctx, lambda: call(q), lambda: call(q + 4))
    for p in (kc, vc, table, q, gate, out, part):
        ctx.free(p)


def weights(ctx, K, R):
    w = ga.Q2W()
    ctx.gd_q2w_alloc(K, R, C.byref(w))
    ctx.gd_rand_q2w(C.byref(w), 5, 0.01, 0.05)
    return w


@pytest.mark.parametrize("T,K,ff", [(2, 128, 17408), (8, 256, 8192), (8, 384, 34816), (17, 640, 12288),
                                    (32, 1024, 34816), (2, 2048, 34816), (27, 5120, 17408), (32, 2048, 6144)])
def test_swiglu_few_tokens(ctx, T, K, ff):
    """Few tokens at every K and ff against the tiles, which a forced plan takes."""
    w, x, o = weights(ctx, K, 2 * ff), zeros(ctx, T * K * 2), zeros(ctx, T * ff * 2)
    not_slower(ctx, lambda: ctx.gd_q2_0_gemm_swiglu(C.byref(w), T, x, o),
               lambda: ctx.gd_q2_0_gemm_swiglu_plan(C.byref(w), T, x, o, 0), 20)
    ctx.gd_q2w_free(C.byref(w))
    for p in (x, o):
        ctx.free(p)


@pytest.mark.parametrize("T,K,R", [(2, 128, 1024), (8, 128, 12288), (32, 256, 16384), (8, 256, 4096), (17, 384, 16384), (27, 5120, 5120)])
def test_gemm_few_tokens_plan(ctx, T, K, R):
    """Few tokens at every K against a tile that needs no K split."""
    w, x, o = weights(ctx, K, R), zeros(ctx, T * K * 2), zeros(ctx, T * R * 4)
    not_slower(ctx, lambda: ctx.gd_q2_0_gemm(C.byref(w), T, x, ga.F16, o, ga.F32),
               lambda: ctx.gd_q2_0_gemm_plan(C.byref(w), T, x, ga.F16, o, ga.F32, 1, 1, 1, 4), 20)
    ctx.gd_q2w_free(C.byref(w))
    for p in (x, o):
        ctx.free(p)
