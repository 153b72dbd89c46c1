"""The framework's work, as cases that can be timed and compared.

Each kind of case is one thing a host program has the library do through its
C ABI (include/gadeon_hip.h): single kernels as MetalEnc's callers use them,
the blocks of a layer, and whole model calls.  `prepare` makes what such a
program holds before the call (weights, caches, states, buffers and the
argument list of every call), `run` makes the calls, `exact` restates them in
64 bits with plain torch.

Sizes: the stack's own geometries (the hybrid of hidden 5120 with 40/8
attention heads of 128 and 16/16 GDN heads, its 48/16-head GDN and 24/4 x 256
attention variants, the dense 1.7B lineage), over prompts, contexts and batch
sizes from the smallest to the largest those geometries are served at.
"""
from __future__ import annotations

import ctypes as C
import math
import weakref

import numpy as np
import torch

import gadeon_amd as ga

F32, F16 = ga.F32, ga.F16
EPS = 1e-6
PAGE = 16                        # positions of a KV page, as the stack uses

HYBRID = dict(n_layer=4, n_embd=5120, n_ff=17408, n_head=40, n_head_kv=8, head_dim=128,
              n_rot=64, rope_base=1e7, eps=EPS, n_vocab=151936, attn_interval=4, d_state=128,
              n_k_head=16, n_v_head=16, d_conv=4, kv_block=PAGE, dense=0)
DENSE = dict(n_layer=4, n_embd=2048, n_ff=6144, n_head=16, n_head_kv=8, head_dim=128,
             n_rot=128, rope_base=1e6, eps=EPS, n_vocab=151936, attn_interval=1, d_state=0,
             n_k_head=0, n_v_head=0, d_conv=0, kv_block=PAGE, dense=1)

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # Decode: the smallest projection of a layer, where the launch counts.
        dict(name="gemv_small", kind="gemv", K=1024, R=3072, x="f16"),
        # Decode: the logits of one token; x in the f32 the reference's buffers hold.
        dict(name="gemv_lm_head", kind="gemv", K=5120, R=151936, x="f32"),
        # A short chat turn appended to a long history.
        dict(name="gemm_turn", kind="gemm", T=27, K=5120, R=17408, x="f32", y="f32"),
        # One prompt chunk through an up projection.
        dict(name="gemm_prompt", kind="gemm", T=512, K=5120, R=17408, x="f16", y="f16"),
        # The feed-forward block on a ragged prompt: norm, SwiGLU GEMM, down GEMM, residual.
        dict(name="mlp_ragged", kind="mlp", T=333, E=5120, FF=17408),
        # The recurrence over one prompt chunk.
        dict(name="gdn_scan", kind="gdn_scan", T=512, nV=16, nK=16, x="f16", chunk=64),
        # The GDN layer between its projections, one entry per operation as the
        # engine encodes it: gate, conv, norms, scan, gated norm; ragged length.
        dict(name="gdn_layer", kind="gdn_layer", T=1000, nV=48, nK=16),
        # Serving: one token of 32 independent sequences.
        dict(name="gdn_step_batch", kind="gdn_step", B=32, nV=16, nK=16, x="f16", gate=True),
        # A later chunk of a long prompt: append K and V, attend to the history.
        dict(name="attn_chunk", kind="attn_prompt", T=512, base=3584, H=40, HKV=8, hd=128, gated=True),
        # One token at a long context: append, attend.
        dict(name="attn_long_token", kind="attn_token", T=9001, H=24, HKV=4, hd=256, gated=True),
        # Whole calls: a prompt chunk to logits, and tokens decoded one at a time.
        dict(name="model_prompt", kind="model_prompt", arch="hybrid", T=512),
        dict(name="model_decode", kind="model_decode", arch="hybrid", P=700, steps=8),
    ]


def _spread(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    k128 = lambda lo, hi: 128 * _spread(rng, lo // 128, hi // 128)  # noqa: E731
    kind = rng.choice(["gemv", "gemm", "mlp", "gdn_scan", "gdn_layer", "gdn_step", "attn_prompt",
                       "attn_token", "model_prompt", "model_decode"])
    heads = lambda: rng.choice([(16, 16), (48, 16), (32, 16), (16, 8)])  # noqa: E731
    att = lambda: dict(zip(("H", "HKV", "hd", "gated"), rng.choice(  # noqa: E731
        [(40, 8, 128, True), (24, 4, 256, True), (16, 8, 128, False)])))
    if kind == "gemv":
        return dict(kind=kind, K=k128(512, 17408), R=_spread(rng, 256, 151936), x=rng.choice(["f16", "f32"]))
    if kind == "gemm":
        K, R = k128(1024, 17408), _spread(rng, 1024, 34816)
        T = min(_spread(rng, 2, 2048), int(5e11 / (K * R)))
        return dict(kind=kind, T=T, K=K, R=R, x=rng.choice(["f16", "f32"]), y=rng.choice(["f16", "f32"]))
    if kind == "mlp":
        return dict(kind=kind, T=_spread(rng, 2, 1024), E=k128(1024, 5120), FF=k128(3072, 17408))
    if kind == "gdn_scan":
        nV, nK = heads()
        return dict(kind=kind, T=_spread(rng, 16, 4096), nV=nV, nK=nK, x=rng.choice(["f16", "f32"]),
                    chunk=rng.choice([32, 64]))
    if kind == "gdn_layer":
        nV, nK = heads()
        return dict(kind=kind, T=_spread(rng, 2, 2048), nV=nV, nK=nK)
    if kind == "gdn_step":
        nV, nK = heads()
        return dict(kind=kind, B=_spread(rng, 1, 64), nV=nV, nK=nK, x=rng.choice(["f16", "f32"]),
                    gate=rng.choice([True, False]))
    if kind == "attn_prompt":
        return dict(kind=kind, T=_spread(rng, 2, 1024), base=rng.choice([0, _spread(rng, 16, 4096)]), **att())
    if kind == "attn_token":
        return dict(kind=kind, T=_spread(rng, 16, 32768), **att())
    arch = rng.choice(["hybrid", "dense"])
    if kind == "model_prompt":
        return dict(kind=kind, arch=arch, T=_spread(rng, 2, 512))
    return dict(kind=kind, arch=arch, P=_spread(rng, 16, 2000), steps=rng.randint(2, 8))


# ------------------------------------------------------------------ inputs

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = ga.Context(0)
    return _ctx


class _Draw:
    """Seeded draws on the GPU: the same sequence for prepare and exact."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * std).to(dtype)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def weights(self, K, R):
        """Ternary codes 0..2 [R][K] and f16 scales [R][K / 128]."""
        codes = torch.randint(0, 3, (R, K), generator=self.g, device="cuda", dtype=torch.uint8)
        return codes, self.uniform(0.01, 0.05, R, K // 128).half()

    def table(self, pages):
        return torch.randperm(pages, generator=self.g, device="cuda").int()


def _dt(name):
    return (F16, torch.float16) if name == "f16" else (F32, torch.float32)


def _dense64(codes, scales):
    R, K = codes.shape
    w = (codes.double() - 1).view(R, K // 128, 128) * scales.double()[:, :, None]
    return w.view(R, K)


class _Weights:
    """A device Q2_0 matrix repacked from GGUF blocks, freed with this object."""

    def __init__(self, codes, scales):
        R, K = codes.shape
        c = codes.view(R * K // 128, 32, 4)
        q = c[..., 0] | c[..., 1] << 2 | c[..., 2] << 4 | c[..., 3] << 6
        gguf = torch.cat([scales.reshape(-1, 1).view(torch.uint8), q], 1).contiguous()
        ctx, self.w = _context(), ga.Q2W()
        ctx.gd_q2w_alloc(K, R, C.byref(self.w))
        weakref.finalize(self, ctx.lib.gd_q2w_free, ctx.h, C.pointer(self.w))
        torch.cuda.synchronize()                 # the blocks were made on torch's stream
        ctx.gd_q2_0_repack(gguf.data_ptr(), 0, C.byref(self.w))
        ctx.sync()
        self.ref = C.byref(self.w)


def _arg(a):
    return a.data_ptr() if isinstance(a, torch.Tensor) else a


def _program(calls, out, keep):
    """The calls a program makes in a pass, with their arguments in hand."""
    ctx = _context()
    torch.cuda.synchronize()
    return {"calls": [(getattr(ctx.lib, name), [ctx.h] + [_arg(a) for a in args]) for name, *args in calls],
            "out": out, "keep": (keep, calls)}


def run(state):
    for fn, args in state["calls"]:
        rc = fn(*args)
        if rc:
            raise RuntimeError(_context().lib.gd_last_error(_context().h).decode())
    return state["out"]


def _new(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _gdn_inputs(r, case, T):
    """q, k L2-normalized, v, log decay, beta and the state of one recurrence."""
    nV, nK, (_, dt) = case["nV"], case["nK"], _dt(case["x"])
    q, k = (torch.nn.functional.normalize(r.normal(T, nK, 128), dim=-1).to(dt) for _ in range(2))
    v = r.normal(T, nV, 128, dtype=dt)
    g, beta = -torch.nn.functional.softplus(r.normal(T, nV)), torch.sigmoid(r.normal(T, nV))
    return q, k, v, g, beta, r.normal(nV, 128, 128, std=0.02)


def _layer_inputs(r, case):
    """A GDN layer's projection rows and parameters, and its states."""
    T, nV, nK = case["T"], case["nV"], case["nK"]
    cd = 128 * (2 * nK + nV)
    return dict(x=r.normal(T, cd), z=r.normal(T, nV * 128), b=r.normal(T, nV), a=r.normal(T, nV),
                dt=r.uniform(-0.5, 0.5, nV), an=r.uniform(-2, -0.3, nV), cw=r.uniform(-0.5, 0.5, cd, 4),
                w=r.uniform(0.8, 1.2, 128), ring=r.normal(3, cd), S=r.normal(nV, 128, 128, std=0.02))


def _step_inputs(r, case):
    B, nV, nK, (_, dt) = case["B"], case["nV"], case["nK"], _dt(case["x"])
    q, k, v = r.normal(B, nK, 128, dtype=dt), r.normal(B, nK, 128, dtype=dt), r.normal(B, nV, 128, dtype=dt)
    g, b = r.normal(B, nV), r.normal(B, nV)
    d, an = r.uniform(-0.5, 0.5, nV), r.uniform(-2, -0.3, nV)
    if not case["gate"]:
        g, b = -torch.nn.functional.softplus(g), torch.sigmoid(b)
    return q, k, v, g, b, d, an, r.normal(B, nV, 128, 128, std=0.02)


def _attn_inputs(r, case):
    """Queries, gates, new K and V, and a cache of shuffled pages.  Normed
    queries and keys, as the layer's q and k norms leave them."""
    n, H, HKV, hd = (1 if case["kind"] == "attn_token" else case["T"]), case["H"], case["HKV"], case["hd"]
    total = case["T"] if case["kind"] == "attn_token" else case["base"] + case["T"]
    pages = -(-total // PAGE) + 1
    q, gate = r.normal(n, H, hd), r.normal(n, H, hd)
    k, v = r.normal(n, HKV, hd), r.normal(n, HKV, hd)
    kc, vc = (r.normal(pages, PAGE, HKV, hd, dtype=torch.float16) for _ in range(2))
    return q, gate, k, v, kc, vc, r.table(pages), n, total


def _model(case):
    cfg = dict(HYBRID if case["arch"] == "hybrid" else DENSE)
    n = case["T"] if case["kind"] == "model_prompt" else case["P"] + case["steps"]
    cfg.update(max_ctx=n, max_batch=512)
    return cfg, n


def _ids(case, seed, n):
    return np.random.default_rng(seed).integers(0, 151936, n).astype(np.int32)


def prepare(case, seed):
    ctx, r, kind = _context(), _Draw(seed), case["kind"]
    if kind == "gemv":
        code, dt = _dt(case["x"])
        w, x, y = _Weights(*r.weights(case["K"], case["R"])), r.normal(case["K"], dtype=dt), _new(case["R"])
        return _program([("gd_q2_0_gemv", w.ref, x, code, y)], y, w)
    if kind == "gemm":
        (xc, xd), (yc, yd) = _dt(case["x"]), _dt(case["y"])
        w, x = _Weights(*r.weights(case["K"], case["R"])), r.normal(case["T"], case["K"], dtype=xd)
        y = _new(case["T"], case["R"], dtype=yd)
        return _program([("gd_q2_0_gemm", w.ref, case["T"], x, xc, y, yc)], y, w)
    if kind == "mlp":
        T, E, FF = case["T"], case["E"], case["FF"]
        gu, down = _Weights(*r.weights(E, 2 * FF)), _Weights(*r.weights(FF, E))
        x, nw = r.normal(T, E), r.uniform(0.8, 1.2, E)
        xn, a, y = _new(T, E, dtype=torch.float16), _new(T, FF, dtype=torch.float16), _new(T, E)
        return _program([("gd_rmsnorm", x, nw, xn, F16, E, T, EPS), ("gd_q2_0_gemm_swiglu", gu.ref, T, xn, a),
                         ("gd_q2_0_gemm", down.ref, T, a, F16, y, F32), ("gd_add", y, x, T * E)], y, (gu, down))
    if kind == "gdn_scan":
        T, nV, nK, (code, dt) = case["T"], case["nV"], case["nK"], _dt(case["x"])
        q, k, v, g, beta, S = _gdn_inputs(r, case, T)
        o = _new(T, nV, 128, dtype=dt)
        return _program([("gd_gdn_prefill", T, nV, nK, 128, 128, q, nK * 128, k, nK * 128, v, nV * 128, code,
                          g, beta, S, o, nV * 128, code, 128 ** -0.5, case["chunk"])], [o, S], None)
    if kind == "gdn_layer":
        T, nV, nK, i = case["T"], case["nV"], case["nK"], _layer_inputs(r, case)
        kd, vd = 128 * nK, 128 * nV
        cd = 2 * kd + vd
        beta, g, conv, o = _new(T, nV), _new(T, nV), _new(T, cd), _new(T, vd)
        return _program([("gd_gdn_gate", i["b"], i["a"], i["dt"], i["an"], beta, g, nV, T * nV),
                         ("gd_gdn_conv", i["x"], i["ring"], i["cw"], conv, cd, 4, T),
                         ("gd_l2norm_rows", conv, 128, 2 * nK, cd, T, EPS),
                         ("gd_gdn_scan_batch", conv, kd, vd, cd, g, beta, i["S"], o, nV, nK, 128, 128 ** -0.5, T),
                         ("gd_rmsnorm_rows", o, 128, T * nV, i["w"], EPS), ("gd_mul_silu", o, i["z"], T * vd)],
                        [o, i["S"], i["ring"]], i)
    if kind == "gdn_step":
        B, nV, nK, (code, dt) = case["B"], case["nV"], case["nK"], _dt(case["x"])
        q, k, v, g, b, d, an, S = _step_inputs(r, case)
        o, fused = _new(B, nV, 128, dtype=dt), case["gate"]
        return _program([("gd_gdn_decode", B, nV, nK, 128, q, k, v, code, g, b, d if fused else None,
                          an if fused else None, S, o, 128 ** -0.5, EPS)], [o, S], None)
    if kind in ("attn_prompt", "attn_token"):
        H, HKV, hd, gated = case["H"], case["HKV"], case["hd"], int(case["gated"])
        q, gate, k, v, kc, vc, table, n, total = _attn_inputs(r, case)
        out, kvd = _new(n, H, hd), HKV * hd
        append = ("gd_kv_append", k, v, kc, vc, table, kvd, total - n, PAGE, n)
        if kind == "attn_prompt":
            attend = ("gd_attn_batch", q, kc, vc, table, gate, out, hd, H, HKV, kvd, PAGE, hd ** -0.5,
                      case["base"], n, gated, 0)
        else:
            attend = ("gd_attn_paged", q, kc, vc, table, gate, out, _new(H * 16 * (hd + 2)), hd, H, HKV, total,
                      kvd, PAGE, hd ** -0.5, gated, 0)
        return _program([append, attend], out, None)
    cfg, n = _model(case)
    st, ids = C.c_void_p(), _ids(case, seed, n)
    ctx.gd_stack_create(C.byref(ga.StackConfig(**cfg)), seed, C.byref(st))
    own = type("Stack", (), {})()
    weakref.finalize(own, ctx.lib.gd_stack_destroy, st)
    nxt, lib = C.c_int32(), ctx.lib
    steps = case.get("steps", 1)
    logits = np.zeros((steps, cfg["n_vocab"]), np.float32)
    if kind == "model_prompt":
        calls = [(lib.gd_stack_reset, [st]),
                 (lib.gd_stack_prefill, [st, ids.ctypes.data, n, C.byref(nxt), logits.ctypes.data])]
    else:
        # A history to return to, and the tokens that follow it.
        P, mark = case["P"], C.c_void_p()
        ctx.check(lib.gd_stack_prefill(st, ids.ctypes.data, P, None, None))
        ctx.check(lib.gd_stack_bookmark(st, C.byref(mark)))
        weakref.finalize(own, lib.gd_bookmark_free, mark)
        calls = [(lib.gd_stack_restore, [st, mark])]
        calls += [(lib.gd_stack_decode, [st, int(ids[P + i]), C.byref(nxt), logits[i].ctypes.data])
                  for i in range(steps)]
    return {"calls": calls, "out": logits, "keep": (own, ids, logits, nxt)}


# ------------------------------------------------------------------ bytes and operations


def _q2(K, R):
    return K * R * 34 / 128


def work(case):
    kind, size = case["kind"], {"f16": 2, "f32": 4}
    if kind == "gemv":
        K, R = case["K"], case["R"]
        return {"bytes": _q2(K, R) + K * size[case["x"]] + 4 * R, "flops": 2 * K * R}
    if kind == "gemm":
        T, K, R = case["T"], case["K"], case["R"]
        return {"bytes": _q2(K, R) + T * (K * size[case["x"]] + R * size[case["y"]]), "flops": 2 * T * K * R}
    if kind == "mlp":
        T, E, FF = case["T"], case["E"], case["FF"]
        return {"bytes": 3 * _q2(E, FF) + T * E * 8 + 4 * E, "flops": 6 * T * E * FF}
    if kind in ("gdn_scan", "gdn_layer"):
        T, nV, nK, z = case["T"], case["nV"], case["nK"], size[case.get("x", "f32")]
        state = 2 * nV * 128 * 128 * 4
        # Rows in and out, the gates; the layer's z and its conv ring and weights too.
        rows = T * (128 * (2 * nK + 2 * nV) * z + 8 * nV)
        if kind == "gdn_layer":
            rows += T * 128 * nV * 4 + 128 * (2 * nK + nV) * (4 + 2 * 3) * 4
        return {"bytes": rows + state, "flops": T * nV * 128 * 128 * 7}
    if kind == "gdn_step":
        B, nV, nK, z = case["B"], case["nV"], case["nK"], size[case["x"]]
        return {"bytes": B * (2 * nV * 128 * 128 * 4 + 128 * (2 * nK + 2 * nV) * z + 8 * nV),
                "flops": B * nV * 128 * 128 * 7}
    if kind in ("attn_prompt", "attn_token"):
        H, HKV, hd = case["H"], case["HKV"], case["hd"]
        n, total = (1, case["T"]) if kind == "attn_token" else (case["T"], case["base"] + case["T"])
        pairs = n * (total - n) + n * (n + 1) / 2
        rows = n * H * hd * 4 * (3 if case["gated"] else 2) + n * HKV * hd * (8 + 4)
        return {"bytes": (total - n) * HKV * hd * 4 + rows, "flops": 4 * pairs * H * hd}
    cfg, n = _model(case)
    E, FF, H, HKV, hd, V = (cfg[k] for k in ("n_embd", "n_ff", "n_head", "n_head_kv", "head_dim", "n_vocab"))
    q = H * hd * (1 if cfg["dense"] else 2)
    att = cfg["n_layer"] // cfg["attn_interval"]
    rec = cfg["n_layer"] - att
    vd = 128 * cfg["n_v_head"]
    cd = 256 * cfg["n_k_head"] + vd
    trunk = att * E * (q + 2 * HKV * hd + H * hd) + rec * E * (cd + 2 * vd + 2 * cfg["n_v_head"])
    trunk += cfg["n_layer"] * 3 * E * FF
    state = rec * 2 * (vd * 128 + 3 * cd) * 4
    passes, first = (1, 0) if kind == "model_prompt" else (case["steps"], case["P"])
    tokens, seen = n - first, sum(range(first + 1, n + 1))
    kv = 4 * HKV * hd * att
    nbytes = passes * (_q2(1, trunk) + _q2(E, V) + 4 * V + state) + tokens * (kv + _q2(1, E)) + (seen if passes > 1 else 0) * kv
    flops = 2 * tokens * trunk + 2 * passes * E * V + 4 * seen * H * hd * att + tokens * rec * vd * 128 * 7
    return {"bytes": nbytes, "flops": flops}


# About four times what the path differs by from the exact result over these
# ranges: f32 sums; the four e4m3 pieces of the GEMV's x (20 bits, groups of 8
# products at 13); the hi + lo f16 operands of attention and the chunked scan
# (22 bits, through the recurrence); operands or outputs rounded to f16; and a
# model's f16 GEMM inputs and KV cache through its layers.
_F16_REL = 1e-3
_TOL = {"gemv": 4e-5, "gemm": _F16_REL, "mlp": 1.5e-3, "gdn_scan": 5e-5, "gdn_layer": 5e-5, "gdn_step": 1e-5,
        "attn_prompt": 1e-5, "attn_token": 1e-5, "model_prompt": 5e-3, "model_decode": 5e-3}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gdn_scan", "gdn_step") and case["x"] == "f16":
        return {"rel": _F16_REL}
    return {"rel": _TOL[kind]}


# ------------------------------------------------------------------ in 64 bits


def _rms(x, w, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _recurrence(q, k, v, g, beta, S):
    """q, k [T][nK][128], v [T][nV][128], S [nV][128][128] (key-major): o and the state."""
    nV, nK, o = v.shape[-2], k.shape[-2], torch.empty_like(v)
    head = torch.arange(nV, device=v.device) % nK
    q, k, gam = q[:, head] * 128 ** -0.5, k[:, head], torch.exp(g)
    for t in range(v.shape[0]):
        S = S * gam[t][:, None, None]
        d = beta[t][:, None] * (v[t] - torch.matmul(k[t][:, None], S)[:, 0])
        S = S + k[t][:, :, None] * d[:, None, :]
        o[t] = torch.matmul(q[t][:, None], S)[:, 0]
    return o, S


def _gdn_rows(x, z, b, a, dt, an, cw, w, ring, S, nV, nK):
    """A GDN layer from its projection rows to its gated output."""
    T, cd = x.shape
    win = torch.cat([ring, x])
    conv = _silu(sum(win[j:j + T] * cw[:, j] for j in range(4)))
    qk = conv[:, :256 * nK].reshape(T, 2 * nK, 128)
    qk = qk / torch.sqrt((qk * qk).sum(-1, keepdim=True) + EPS)
    g = torch.nn.functional.softplus(a + dt) * an
    o, S = _recurrence(qk[:, :nK], qk[:, nK:], conv[:, 256 * nK:].reshape(T, nV, 128), g, torch.sigmoid(b), S)
    return (_rms(o, w) * _silu(z.reshape(T, nV, 128))).reshape(T, nV * 128), S, win[T:]


def _attend(q, k, v, first, hd):
    """q [n][H][hd] at positions first .., k and v [total][HKV][hd]."""
    n, H, total, HKV = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    seen = torch.arange(total, device=q.device)[None] <= first + torch.arange(n, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(H):
        s = (q[:, h] @ k[:, h * HKV // H].T) * hd ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, h * HKV // H]
    return out


def _lcg(seed, n):
    """The library's counter-addressable LCG stream: its first n 31-bit values."""
    wrap = lambda x: (x + 2 ** 63) % 2 ** 64 - 2 ** 63  # noqa: E731
    a, c = 6364136223846793005, 1442695040888963407
    s = torch.empty(n, dtype=torch.int64, device="cuda")
    s[0] = wrap((seed + 0x9E3779B97F4A7C15) * a + c)
    m = 1
    while m < n:                                 # the map of m steps doubles the known prefix
        s[m:2 * m] = s[:min(m, n - m)] * wrap(a) + wrap(c)
        a, c, m = a * a % 2 ** 64, (a * c + c) % 2 ** 64, 2 * m
    return (s >> 33) & 0x7FFFFFFF


def _lcg_uniform(seed, n, lo, hi):
    lo, span = np.float32(lo), np.float32(hi) - np.float32(lo)
    return _lcg(seed, n).float() * 2.0 ** -31 * float(span) + float(lo)


def _rotate(x, n_rot, base):
    """Partial NEOX rope of x [T][heads][hd] at positions 0 .. T-1."""
    half = n_rot // 2
    f = base ** (-torch.arange(half, dtype=torch.float64, device=x.device) * 2 / n_rot)
    ang = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None, None] * f
    a, b = x[..., :half], x[..., half:n_rot]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos(), x[..., n_rot:]], -1)


def _forward(cfg, seed, ids, last):
    """Logits of the last positions of ids, the weights drawn as the stack draws them."""
    sd = seed * 1000003 % 2 ** 64

    def nxt():
        nonlocal sd
        sd += 2
        return sd

    def matrix(K, R):
        s = nxt()
        codes = ((_lcg(s, K * R) * 3) >> 31).to(torch.uint8).view(R, K)
        return _dense64(codes, _lcg_uniform(s + 1, K * R // 128, 0.01, 0.05).half().view(R, K // 128))

    vec = lambda n, lo, hi: _lcg_uniform(nxt(), n, lo, hi).double()  # noqa: E731
    E, FF, H, HKV, hd, V = (cfg[k] for k in ("n_embd", "n_ff", "n_head", "n_head_kv", "head_dim", "n_vocab"))
    nV, nK, T = cfg["n_v_head"], cfg["n_k_head"], len(ids)
    # The embedding is drawn after every layer: skip ahead to it first.
    rec = [(il + 1) % cfg["attn_interval"] != 0 for il in range(cfg["n_layer"])]
    start = sd
    sd += 2 * sum(10 if r else 8 for r in rec)
    embd, out_norm = matrix(E, V), vec(E, 0.8, 1.2)
    x = embd[torch.from_numpy(ids).long().cuda()]
    sd = start
    for is_rec in rec:
        an, pn = vec(E, 0.8, 1.2), vec(E, 0.8, 1.2)
        n = _rms(x, an)
        if is_rec:
            cd, vd = 128 * (2 * nK + nV), 128 * nV
            proj = n @ matrix(E, cd + vd + 2 * nV).T
            out = matrix(vd, E)
            cw, dt, aneg = vec(cd * 4, -0.5, 0.5).view(cd, 4), vec(nV, -0.5, 0.5), vec(nV, -2, -0.3)
            a = _gdn_rows(proj[:, :cd], proj[:, cd:cd + vd], proj[:, cd + vd:cd + vd + nV], proj[:, cd + vd + nV:],
                          dt, aneg, cw, vec(128, 0.8, 1.2), n.new_zeros(3, cd), n.new_zeros(nV, 128, 128), nV, nK)[0]
        else:
            qs = 1 if cfg["dense"] else 2
            proj = n @ matrix(E, (qs * H + 2 * HKV) * hd).T
            out, qn, kn = matrix(H * hd, E), vec(hd, 0.8, 1.2), vec(hd, 0.8, 1.2)
            q = proj[:, :qs * H * hd].view(T, H, qs * hd)
            k, v = proj[:, qs * H * hd:].view(T, 2, HKV, hd).unbind(1)
            rot = lambda y, w: _rotate(_rms(y, w), cfg["n_rot"], cfg["rope_base"])  # noqa: E731
            a = _attend(rot(q[..., :hd], qn), rot(k, kn), v, 0, hd)
            a = (a if cfg["dense"] else a * torch.sigmoid(q[..., hd:])).reshape(T, H * hd)
        x = x + a @ out.T
        del out
        gu = _rms(x, pn) @ matrix(E, 2 * FF).T
        x = x + (_silu(gu[:, :FF]) * gu[:, FF:]) @ matrix(FF, E).T
    return _rms(x[-last:], out_norm) @ embd.T


def exact(case, seed):
    r, kind = _Draw(seed), case["kind"]
    if kind in ("gemv", "gemm"):
        w = _dense64(*r.weights(case["K"], case["R"]))
        dt = _dt(case["x"])[1]
        if kind == "gemv":
            return w @ r.normal(case["K"], dtype=dt).double()
        return r.normal(case["T"], case["K"], dtype=dt).double() @ w.T
    if kind == "mlp":
        T, E, FF = case["T"], case["E"], case["FF"]
        gu, down = _dense64(*r.weights(E, 2 * FF)), _dense64(*r.weights(FF, E))
        x, nw = r.normal(T, E).double(), r.uniform(0.8, 1.2, E).double()
        h = _rms(x, nw) @ gu.T
        return (_silu(h[:, :FF]) * h[:, FF:]) @ down.T + x
    if kind == "gdn_scan":
        return list(_recurrence(*(t.double() for t in _gdn_inputs(r, case, case["T"]))))
    if kind == "gdn_layer":
        i = {k: v.double() for k, v in _layer_inputs(r, case).items()}
        return list(_gdn_rows(i["x"], i["z"], i["b"], i["a"], i["dt"], i["an"], i["cw"], i["w"], i["ring"], i["S"],
                              case["nV"], case["nK"]))
    if kind == "gdn_step":
        q, k, v, g, b, d, an, S = (t.double() for t in _step_inputs(r, case))
        if case["gate"]:
            g, b = torch.nn.functional.softplus(g + d) * an, torch.sigmoid(b)
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + EPS) for t in (q, k))
        got = [_recurrence(q[i:i + 1], k[i:i + 1], v[i:i + 1], g[i:i + 1], b[i:i + 1], S[i]) for i in range(len(q))]
        return [torch.cat([o for o, _ in got]), torch.stack([s for _, s in got])]
    if kind in ("attn_prompt", "attn_token"):
        q, gate, k, v, kc, vc, table, n, total = _attn_inputs(r, case)
        # New keys and values enter as the cache holds them: the f16 values are the inputs of the attention.
        rows = lambda c, new: torch.cat([c[table.long()].flatten(0, 1)[:total - n], new.half()]).double()  # noqa: E731
        out = _attend(q.double(), rows(kc, k), rows(vc, v), total - n, case["hd"])
        return out * torch.sigmoid(gate.double()) if case["gated"] else out
    cfg, n = _model(case)
    return _forward(cfg, seed, _ids(case, seed, n), case.get("steps", 1))
