"""The attention entries of the C ABI (gd_split_q_gate, gd_rope, gd_kv_append,
gd_attn_paged, gd_attn_batch; MetalEnc.swift:656-706, 780-847, 966-1025)
against an f64 restatement of Attn.step's attention (Attention.swift:79-134):
q and k RMS-normalized and rotated by the oracle's Kern.ropeNeox, K and V
rounded to f16 as the cache holds them, softmax((q . k) / sqrt(hd)) . v, times
sigmoid(gate).  Head dims 128 and 256 with the GQA groups of BASELINE config 4
(40 / 8) and of the reference's 27B (24 / 4), over ragged page sizes.  Norm-wise
relative error < 2e-3 (the f16 cache and the hi/lo f16 MFMA operands are the
error sources); rope and the q|gate split against the oracle / exactly; the
cache append bit-exact (RNE f16).  Prompts up to 600 keys (many query
blocks, dispatched longest first): rows of every query block are checked, and
a second launch of the same call is bit-identical."""
import ctypes as C

import numpy as np
import pytest

import gadeon_amd as ga
import oracle as O
from conftest import rel_diff

pytestmark = pytest.mark.gpu
TOL = 2e-3


def sigmoid(x):
    return 1.0 / (1.0 + np.exp(-x))


def make_cache(ctx, T, kv_dim, page, seed):
    """A pool of pages in shuffled order (the table maps positions to pages)."""
    npages = (T + page - 1) // page + 2
    rng = np.random.default_rng(seed)
    table = rng.permutation(npages).astype(np.int32)
    kc = ctx.alloc(npages * page * kv_dim * 2)
    vc = ctx.alloc(npages * page * kv_dim * 2)
    ctx.gd_fill_u32(kc, 0x7e007e00, npages * page * kv_dim // 2)     # f16 NaN: unread
    ctx.gd_fill_u32(vc, 0x7e007e00, npages * page * kv_dim // 2)
    return kc, vc, ctx.put(table), table, npages


def ref_attention(q, K, V, gate, nkv, t_end):
    """q [nh][hd] at the keys 0 .. t_end-1 of K, V [T][nkv][hd] (f64)."""
    nh, hd = q.shape
    grp = nh // nkv
    out = np.empty((nh, hd))
    for h in range(nh):
        k = K[:t_end, h // grp].astype(np.float64)
        v = V[:t_end, h // grp].astype(np.float64)
        s = k @ q[h].astype(np.float64) / np.sqrt(hd)
        p = np.exp(s - s.max())
        out[h] = (p / p.sum()) @ v * sigmoid(gate[h].astype(np.float64))
    return out


@pytest.mark.parametrize("hd,nh,nkv,page,T", [(128, 40, 8, 16, 77), (256, 24, 4, 16, 130),
                                              (256, 24, 4, 7, 45), (128, 4, 2, 5, 300),
                                              (128, 40, 8, 16, 600), (256, 24, 4, 16, 520)])
def test_decode_and_batch_attention(ctx, hd, nh, nkv, page, T):
    rng = np.random.default_rng(hd + T)
    kv_dim = hd * nkv
    n_rot, base, eps = 64, 1e7, 1e-6
    # Projections as the engine makes them: per head q | gate, then norms, rope.
    qfull = rng.standard_normal((T, nh, 2 * hd)).astype(np.float32)
    k = rng.standard_normal((T, nkv, hd)).astype(np.float32)
    v = rng.standard_normal((T, nkv, hd)).astype(np.float32)
    qn = rng.uniform(0.8, 1.2, hd).astype(np.float32)
    kn = rng.uniform(0.8, 1.2, hd).astype(np.float32)
    # device: split, norm, rope, append
    dqf = ctx.put(qfull)
    dq, dg = ctx.alloc(T * nh * hd * 4), ctx.alloc(T * nh * hd * 4)
    ctx.gd_split_q_gate(dqf, dq, dg, hd, nh, T)
    q_dev = ctx.get(dq, (T, nh, hd), np.float32)
    assert np.array_equal(q_dev, qfull[:, :, :hd]) and \
        np.array_equal(ctx.get(dg, (T, nh, hd), np.float32), qfull[:, :, hd:])
    dqn, dkn = ctx.put(qn), ctx.put(kn)
    dk, dv = ctx.put(k), ctx.put(v)
    ctx.gd_rmsnorm_rows(dq, hd, T * nh, dqn, eps)
    ctx.gd_rmsnorm_rows(dk, hd, T * nkv, dkn, eps)
    ctx.gd_rope(dq, hd, nh, n_rot, base, 0, T)
    ctx.gd_rope(dk, hd, nkv, n_rot, base, 0, T)
    # oracle: the same preparation per token (Attention.swift:94-107)
    q_ref = np.stack([O.rope_neox(O.rmsnorm_rows(qfull[t, :, :hd].ravel(), hd, qn, eps), hd, n_rot,
                                  base, t) for t in range(T)]).reshape(T, nh, hd)
    k_ref = np.stack([O.rope_neox(O.rmsnorm_rows(k[t].ravel(), hd, kn, eps), hd, n_rot, base, t)
                      for t in range(T)]).reshape(T, nkv, hd)
    # The rotation angle pos * theta carries f32 rounding that grows with the
    # position (about 600 * 2^-24 rad at T = 600): the bound follows it.
    rtol = 1e-5 if T <= 300 else 1e-4
    assert rel_diff(ctx.get(dq, (T, nh, hd), np.float32), q_ref) < rtol
    assert rel_diff(ctx.get(dk, (T, nkv, hd), np.float32), k_ref) < rtol
    kc, vc, dtab, table, npages = make_cache(ctx, T, kv_dim, page, hd)
    # append in two calls (a prefix, then the rest)
    cut = T // 3
    ctx.gd_kv_append(dk, dv, kc, vc, dtab, kv_dim, 0, page, cut)
    ctx.gd_kv_append(dk + cut * kv_dim * 4, dv + cut * kv_dim * 4, kc, vc, dtab, kv_dim, cut, page,
                     T - cut)
    kpool = ctx.get(kc, (npages, page, kv_dim), np.float16)
    vpool = ctx.get(vc, (npages, page, kv_dim), np.float16)
    pos = np.arange(T)
    K16 = kpool[table[pos // page], pos % page].reshape(T, nkv, hd)
    V16 = vpool[table[pos // page], pos % page].reshape(T, nkv, hd)
    k_dev = ctx.get(dk, (T, nkv, hd), np.float32)
    assert np.array_equal(K16, k_dev.astype(np.float16))
    assert np.array_equal(V16, v.astype(np.float16))
    gate = qfull[:, :, hd:]
    # batch (prefill) attention of every token, in two chunks
    dout = ctx.alloc(T * nh * hd * 4)
    scale = 1 / np.sqrt(hd)
    for lo, hi in ((0, cut), (cut, T)):
        ctx.gd_attn_batch(dq + lo * nh * hd * 4, kc, vc, dtab, dg + lo * nh * hd * 4,
                          dout + lo * nh * hd * 4, hd, nh, nkv, kv_dim, page, C.c_float(scale), lo,
                          hi - lo, 1, 0)
    got = ctx.get(dout, (T, nh, hd), np.float32)
    q_used = ctx.get(dq, (T, nh, hd), np.float32)
    for t in sorted({0, 1, cut - 1, cut, T // 2, T - 1, *range(5, T, 61)}):
        want = ref_attention(q_used[t], K16, V16, gate[t], nkv, t + 1)
        assert rel_diff(got[t], want) < TOL, t
    # The same launch again: bit-identical.
    ctx.gd_attn_batch(dq + cut * nh * hd * 4, kc, vc, dtab, dg + cut * nh * hd * 4,
                      dout + cut * nh * hd * 4, hd, nh, nkv, kv_dim, page, C.c_float(scale), cut,
                      T - cut, 1, 0)
    assert np.array_equal(ctx.get(dout, (T, nh, hd), np.float32), got)
    # decode attention of the last token over all T cached keys, gated and not
    part = ctx.alloc(nh * 16 * (hd + 2) * 4)
    dq1 = dq + (T - 1) * nh * hd * 4
    dg1 = dg + (T - 1) * nh * hd * 4
    do1 = ctx.alloc(nh * hd * 4)
    for gated in (1, 0):
        ctx.gd_attn_paged(dq1, kc, vc, dtab, dg1 if gated else None, do1, part, hd, nh, nkv, T,
                          kv_dim, page, C.c_float(scale), gated, 0)
        g1 = gate[T - 1] if gated else np.full((nh, hd), 1e9, np.float32)
        want = ref_attention(q_used[T - 1], K16, V16, g1, nkv, T)
        r = rel_diff(ctx.get(do1, (nh, hd), np.float32), want)
        assert r < TOL, (gated, r)
    # and it equals the batch path's last row
    ctx.gd_attn_paged(dq1, kc, vc, dtab, dg1, do1, part, hd, nh, nkv, T, kv_dim, page,
                      C.c_float(scale), 1, 0)
    assert rel_diff(ctx.get(do1, (nh, hd), np.float32), got[T - 1]) < TOL
    for p in (dqf, dq, dg, dqn, dkn, dk, dv, kc, vc, dtab, dout, part, do1):
        ctx.free(p)


@pytest.mark.parametrize("hd,nh,nkv,page,T,lo", [
    (128, 40, 8, 16, 1, 0), (256, 24, 4, 16, 33, 0), (128, 2, 2, 5, 31, 30), (256, 9, 1, 16, 64, 1),
    (128, 16, 8, 16, 576, 0), (128, 40, 8, 16, 577, 0), (256, 9, 1, 16, 1155, 1), (128, 5, 1, 3, 2047, 0),
    (128, 34, 2, 16, 4099, 0), (256, 6, 1, 7, 4097, 100), (128, 16, 8, 16, 9000, 4999)])
def test_decode_attention_key_blocks(ctx, hd, nh, nkv, page, T, lo):
    """One query over cached keys lo .. T-1 around the edges of the key blocks
    and splits (one key, one past a block, several rounds of a wave) and of the
    few keys that go a wave a key, with one, two, five, six
    and more than eight q heads a kv head: against f64 over the same f16 cache
    within 3e-6 (22-bit q and weights, f32 sums)."""
    rng = np.random.default_rng(T + nh)
    kv_dim, npages = hd * nkv, (T + page - 1) // page + 1
    table = rng.permutation(npages).astype(np.int32)
    K, V = (rng.standard_normal((npages, page, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.standard_normal((nh, hd)).astype(np.float32) for _ in range(2))
    bufs = [ctx.put(a) for a in (q, K.view(np.uint16), V.view(np.uint16), table, gate)]
    out, part = ctx.alloc(nh * hd * 4), ctx.alloc(nh * 16 * (hd + 2) * 4)
    ctx.gd_attn_paged(*bufs, out, part, hd, nh, nkv, T, kv_dim, page, C.c_float(1 / np.sqrt(hd)), 1, lo)
    rows = lambda a: a[table].reshape(npages * page, nkv, hd)[lo:T]
    want = ref_attention(q, rows(K), rows(V), gate, nkv, T - lo)
    assert rel_diff(ctx.get(out, (nh, hd), np.float32), want) < 3e-6
    for p in (*bufs, out, part):
        ctx.free(p)


@pytest.mark.parametrize("hd,nh,nkv,page,T,lo", [
    (128, 24, 4, 16, 768, 0), (128, 24, 4, 16, 769, 0), (128, 6, 6, 16, 1153, 0), (128, 34, 2, 16, 577, 0),
    (256, 24, 4, 16, 1153, 0), (256, 24, 4, 16, 1152, 0), (256, 12, 6, 16, 3585, 0), (256, 12, 4, 5, 1300, 19),
    (256, 3, 1, 16, 2050, 1), (256, 9, 9, 16, 8193, 0), (256, 5, 5, 16, 4097, 0)])
def test_decode_attention_last_few_keys(ctx, hd, nh, nkv, page, T, lo):
    """The last key count that goes a wave a key and the first that does not,
    by the heads and what they share: as test_decode_attention_key_blocks."""
    test_decode_attention_key_blocks(ctx, hd, nh, nkv, page, T, lo)


@pytest.mark.parametrize("hd,nh,nkv", [(128, 10, 2), (256, 6, 1)])
@pytest.mark.parametrize("off", [(4, 0, 0), (0, 4, 0), (0, 0, 4), (8, 8, 8), (0, 0, 0)])
def test_decode_attention_alignment(ctx, hd, nh, nkv, off):
    """q, K or V short of 16-byte alignment (off, bytes), with more keys than
    the few-keys rule takes: the kernel of 16-byte loads is not launched, and
    either kernel's result is within 3e-6 of f64."""
    page, T = 16, 3000
    rng = np.random.default_rng(hd + sum(off))
    kv_dim, npages = hd * nkv, T // page + 1
    table = rng.permutation(npages).astype(np.int32)
    K, V = (rng.standard_normal((npages, page, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.standard_normal((nh, hd)).astype(np.float32) for _ in range(2))
    bufs = [ctx.alloc(a.nbytes + 16) for a in (q, K, V)]
    at = [b + o for b, o in zip(bufs, off)]
    for p, a in zip(at, (q, K.view(np.uint16), V.view(np.uint16))):
        ctx.set(p, a)
    dt, dg = ctx.put(table), ctx.put(gate)
    out, part = ctx.alloc(nh * hd * 4), ctx.alloc(nh * 16 * (hd + 2) * 4)
    ctx.gd_fill_u32(part, 0xffffffff, nh * 16 * (hd + 2))
    ctx.gd_attn_paged(*at, dt, dg, out, part, hd, nh, nkv, T, kv_dim, page, C.c_float(1 / np.sqrt(hd)), 1, 0)
    rows = lambda a: a[table].reshape(npages * page, nkv, hd)[:T]
    want = ref_attention(q, rows(K), rows(V), gate, nkv, T)
    assert rel_diff(ctx.get(out, (nh, hd), np.float32), want) < 3e-6
    # 16-byte loads need aligned inputs: without them the call has to be the
    # wave-a-key kernel's, whose 16 splits a head fill the caller's scratch.
    used = np.isfinite(ctx.get(part, nh * 16 * (hd + 2), np.float32)).all()
    assert used == any(off)
    for p in (*bufs, dt, dg, out, part):
        ctx.free(p)


@pytest.mark.parametrize("hd,nh,nkv", [(128, 10, 2), (256, 6, 1)])
@pytest.mark.parametrize("T", [200, 5003])
def test_decode_attention_infinities(ctx, hd, nh, nkv, T):
    """Infinite cache entries, with few keys and with many (either kernel): an
    infinite V, at a middling key, at one of almost no weight (below 1e-9
    of the largest), at the one key that holds almost all of it (its weight has no
    low half) and at the last key, gives its dim that infinity and leaves the
    others; an infinite K gives a key no weight where its score is -inf, and
    NaN where it is +inf."""
    page = 16
    rng = np.random.default_rng(hd + T)
    kv_dim, npages = hd * nkv, T // page + 1
    table = rng.permutation(npages).astype(np.int32)
    K, V = (rng.standard_normal((npages * page, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.standard_normal((nh, hd)).astype(np.float32) for _ in range(2))
    q[:, 7] = np.where(np.arange(nh) % 3 == 2, -1.0, 1.0)        # the sign of an infinite K's score
    grp, sc = nh // nkv, 1 / np.sqrt(hd)
    for g in range(nkv):                                        # the heavy and the light key
        u = q[g * grp:(g + 1) * grp].mean(0)
        u[7] = 0
        K[150, g], K[90, g] = 12 * u, -6 * u
    for j, d, x in ((60, 3, np.inf), (90, 4, -np.inf), (150, 5, np.inf), (T - 1, 6, -np.inf)):
        V[j, :, d] = x
    K[160, :, 7] = -np.inf
    paged = np.empty((2, npages, page, nkv, hd), np.float16)
    paged[:, table] = np.stack([K, V]).reshape(2, npages, page, nkv, hd)
    bufs = [ctx.put(a) for a in (q, paged[0].view(np.uint16), paged[1].view(np.uint16), table, gate)]
    out, part = ctx.alloc(nh * hd * 4), ctx.alloc(nh * 16 * (hd + 2) * 4)
    ctx.gd_attn_paged(*bufs, out, part, hd, nh, nkv, T, kv_dim, page, C.c_float(sc), 1, 0)
    got = ctx.get(out, (nh, hd), np.float32)
    Kz, Vz = K.copy(), np.where(np.isinf(V), 0, V)
    Kz[160, :, 7] = 0
    for h in range(nh):
        if q[h, 7] < 0:
            assert np.isnan(got[h]).all(), h
            continue
        s = Kz[:T, h // grp].astype(np.float64) @ q[h].astype(np.float64) * sc
        s[160] = -np.inf
        p = np.exp(s - s.max())
        assert p[150] / p.sum() > 0.5 and p[90] / p[150] < 1e-9       # heavy and light
        want = (p / p.sum()) @ Vz[:T, h // grp].astype(np.float64) * sigmoid(gate[h].astype(np.float64))
        assert got[h, 3] == np.inf and got[h, 4] == -np.inf and got[h, 5] == np.inf and got[h, 6] == -np.inf, h
        fin = np.r_[0:3, 7:hd]
        assert rel_diff(got[h, fin], want[fin]) < 3e-6, h
    for p in (*bufs, out, part):
        ctx.free(p)


@pytest.mark.parametrize("hd,nh,nkv,page,N,base", [
    (256, 6, 2, 16, 1, 127), (256, 8, 2, 5, 3, 700), (256, 4, 4, 16, 65, 1000), (256, 4, 1, 16, 200, 0),
    (256, 2, 1, 7, 64, 4100)])
def test_prefill_attention_key_splits(ctx, hd, nh, nkv, page, N, base):
    """Few queries over many cached keys (head dim 256): two splits and the most,
    query blocks that end before the last splits, queries that precede a whole
    split of their block, rows short of a block: against f64 over the same f16
    cache (q and weights split into 22 bits, f32 sums: 1e-5 of the output)."""
    rng = np.random.default_rng(N + base)
    T, kv_dim = N + base, hd * nkv
    npages = (T + page - 1) // page + 1
    table = rng.permutation(npages).astype(np.int32)
    K, V = (rng.standard_normal((npages, page, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.standard_normal((N, nh, hd)).astype(np.float32) for _ in range(2))
    bufs = [ctx.put(a) for a in (q, K.view(np.uint16), V.view(np.uint16), table, gate)]
    out = ctx.alloc(q.nbytes)
    ctx.gd_attn_batch(*bufs, out, hd, nh, nkv, kv_dim, page, C.c_float(1 / np.sqrt(hd)), base, N, 1, 0)
    got = ctx.get(out, q.shape, np.float32)
    rows = lambda a: a[table].reshape(npages * page, nkv, hd)
    Kr, Vr = rows(K), rows(V)
    for n in range(N):
        want = ref_attention(q[n], Kr[:base + n + 1], Vr[:base + n + 1], gate[n], nkv, base + n + 1)
        assert rel_diff(got[n], want) < 1e-5, n
    for p in (*bufs, out):
        ctx.free(p)


@pytest.mark.parametrize("nh,nkv,N,base", [(8, 2, 5, 700), (12, 2, 700, 0)])
def test_prefill_attention_scales(ctx, nh, nkv, N, base):
    """Head dim 256 at a scale whose products with q round, with its keys split
    over the chip (few queries) and not: both halves of q's split belong to one
    value, so rows stay within 1e-5 of f64 (22-bit q and weights, f32 sums)."""
    hd, page, scale = 256, 16, 0.07
    rng = np.random.default_rng(N)
    T, kv_dim = N + base, hd * nkv
    npages = (T + page - 1) // page
    K, V = (rng.standard_normal((npages * page, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.standard_normal((N, nh, hd)).astype(np.float32) for _ in range(2))
    bufs = [ctx.put(a) for a in (q, K.view(np.uint16), V.view(np.uint16), np.arange(npages, dtype=np.int32), gate)]
    out = ctx.alloc(q.nbytes)
    ctx.gd_attn_batch(*bufs, out, hd, nh, nkv, kv_dim, page, C.c_float(scale), base, N, 1, 0)
    got = ctx.get(out, q.shape, np.float32)
    for n in range(0, N, max(1, N // 8)):
        # ref_attention's scale is 1 / sqrt(hd); the entry's is the f32 nearest 0.07.
        want = ref_attention(q[n].astype(np.float64) * float(np.float32(scale)) * np.sqrt(hd), K, V, gate[n], nkv,
                             base + n + 1)
        assert rel_diff(got[n], want) < 1e-5, n
    for p in (*bufs, out):
        ctx.free(p)


def test_recorded_calls_hold_their_memory(ctx):
    """A recording's attention partials are its own and the workspace it used
    stays with it: launched on another context, between that context's own
    calls, after its first context has grown its workspace and is gone, every
    replay of a long-context token, a few-queries prompt and a GEMM of f32 rows
    gives the direct calls' bits."""
    hd, nh, nkv, page, T, N, K, R = 256, 8, 2, 16, 4000, 5, 1024, 512
    rng = np.random.default_rng(3)
    kv_dim, npages = hd * nkv, T // page + 1
    f32 = lambda *s: rng.standard_normal(s).astype(np.float32)
    kc, vc = (ctx.put(f32(npages, page, nkv, hd).astype(np.float16).view(np.uint16)) for _ in range(2))
    q, gate, other, X = (ctx.put(f32(*s)) for s in ((N, nh, hd), (N, nh, hd), (N, nh, hd), (64, K)))
    table = ctx.put(rng.permutation(npages).astype(np.int32))
    w = ga.Q2W()
    blocks = O.lcg_q2_0(K, R, 9)
    ctx.gd_q2_0_upload(blocks.ctypes.data, K, R, C.byref(w))
    outs = [(ctx.alloc(4 * n), n) for n in (nh * hd, N * nh * hd, 8 * R)]
    part, spare = ctx.alloc(nh * 16 * (hd + 2) * 4), ctx.alloc(N * nh * hd * 4)
    ctx.sync()

    def attend(c, src, o1, o2):
        c.gd_attn_paged(src, kc, vc, table, gate, o1, part, hd, nh, nkv, T, kv_dim, page, C.c_float(1 / 16), 1, 0)
        c.gd_attn_batch(src, kc, vc, table, gate, o2, hd, nh, nkv, kv_dim, page, C.c_float(1 / 16), T - N, N, 1, 0)

    def calls(c):
        attend(c, q, outs[0][0], outs[1][0])
        c.gd_q2_0_gemm(C.byref(w), 8, X, ga.F32, outs[2][0], ga.F32)

    first, g = ga.Context(0), C.c_void_p()
    calls(first)
    want = [first.get(p, n, np.float32) for p, n in outs]
    first.gd_graph_begin()
    calls(first)
    first.gd_graph_end(C.byref(g))
    attend(first, other, spare, spare)
    big = first.alloc(64 * R * 4)
    first.gd_q2_0_gemm(C.byref(w), 64, X, ga.F32, big, ga.F32)
    first.close()
    for _ in range(3):
        for p, n in outs:
            ctx.gd_fill_u32(p, 0, n)
        attend(ctx, other, spare, spare)
        ctx.gd_graph_launch(g)
        attend(ctx, other, spare, spare)
        for (p, n), ref in zip(outs, want):
            assert np.array_equal(ctx.get(p, n, np.float32), ref)
    ctx.lib.gd_graph_destroy(g)
    ctx.gd_q2w_free(C.byref(w))
    for p in (kc, vc, q, gate, other, X, table, part, spare, *(p for p, _ in outs)):
        ctx.free(p)


def test_attention_rejects_bad_shapes(ctx):
    d = ctx.alloc(64)
    lib = ctx.lib
    assert lib.gd_attn_paged(ctx.h, d, d, d, d, d, d, d, 64, 4, 2, 8, 128, 16, C.c_float(0.1), 1,
                             0) == ga.GD_EINVAL
    assert b"head_dim" in lib.gd_last_error(ctx.h)
    assert lib.gd_attn_paged(ctx.h, d, d, d, d, d, d, d, 128, 5, 2, 8, 256, 16, C.c_float(0.1), 1,
                             0) == ga.GD_EINVAL
    assert lib.gd_attn_batch(ctx.h, d, d, d, d, d, d, 128, 4, 2, 256, 16, C.c_float(0.1), 0, 4, 1,
                             8) == ga.GD_EINVAL
    assert b"window" in lib.gd_last_error(ctx.h)
    assert lib.gd_rope(ctx.h, d, 128, 2, 130, C.c_float(1e4), 0, 1) == ga.GD_EINVAL
    ctx.free(d)
