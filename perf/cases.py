"""The work that programs built on this library have it do, as cases that can be timed.

Kernel-level cases call the C ABI with torch tensors as device memory, on the
default stream; engine-level cases drive DecodeSession / DecodeBatch. Shapes
are Gemma-3-1B's (hidden 1152, ffn 6912, 4 query heads over 1 KV head of 256,
vocab 262144, a global layer every sixth, window 512), the ones this
repository's benchmark and tests use, and generic ones around them. Weights
are random int4 with N(0, 0.02) group scales, KV rows N(0, 1), as in the
benchmark. exact() is a float64 restatement in plain torch.
"""
import ctypes as C
import math

import numpy as np
import torch

import xpose_amd as X

DEV = "cuda"
HIDDEN, FFN, HEADS, HD, VOCAB = 1152, 6912, 4, 256, 262144
EPS, THETA = 1e-6, {True: 1e6, False: 1e4}
FMT = {"f16": X.XP_SCALE_F16_QUAD, "bf16": X.XP_SCALE_BF16_QUAD, "f32": X.XP_SCALE_F32}
F64 = torch.float64


def listed():
    return [
        # one K or V projection of a decode step: the smallest call, all latency
        {"name": "matvec_kv", "kind": "matvec", "rows": HIDDEN, "cols": 256, "fmt": "f16"},
        # the tied lm_head of a decode step: one long stream of weights
        {"name": "matvec_lm_head", "kind": "matvec", "rows": HIDDEN, "cols": VOCAB, "fmt": "bf16"},
        # a GGUF matrix kept in its own format (Q4_K_M files keep ffn_down so)
        {"name": "native_q4k_down", "kind": "native", "type": "Q4_K", "rows": HIDDEN, "cols": FFN},
        # one decode layer put together from the kernel-level entry points, as
        # an engine with its own scheduler calls them, deep in a context
        {"name": "decode_layer_4000", "kind": "decode_layer", "ctx": 4000, "window": 0, "fmt": "f16"},
        # the attention block of a prompt: a first chunk, and a later chunk of
        # a long one in a sliding-window layer
        {"name": "prefill_attn_200", "kind": "prefill_attention", "tokens": 200, "start": 0, "window": 0},
        {"name": "prefill_attn_1024", "kind": "prefill_attention", "tokens": 1024, "start": 1000,
         "window": 512},
        # drawing a token on the device: over the whole vocabulary, and from its best k
        {"name": "sample_full", "kind": "sample", "vocab": VOCAB, "k": 0, "parts": 4096},
        {"name": "sample_top64", "kind": "sample", "vocab": VOCAB, "k": 64, "parts": 256},
        # whole calls on the full model: the benchmark's short prompt, a long
        # prompt, greedy decode at the headline's context, 16 sequences at once
        {"name": "prefill_32", "kind": "prefill", "layers": 26, "tokens": 32, "start": 0, "fmt": "f16"},
        {"name": "prefill_2000", "kind": "prefill", "layers": 26, "tokens": 2000, "start": 0, "fmt": "f16"},
        {"name": "decode_4096", "kind": "decode", "layers": 26, "ctx": 4096, "steps": 16, "fmt": "f16"},
        {"name": "batch_16", "kind": "batch", "layers": 26, "seqs": 16, "depth": 4096, "steps": 8,
         "fmt": "f16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "native", "decode_layer", "prefill_attention", "prefill_attention", "sample",
                       "prefill", "prefill", "decode", "batch"])
    fmt = rng.choice(["f16", "bf16"])
    if kind == "matvec":
        fmt = rng.choice(["f16", "bf16", "f32"])
        unit = 32 if fmt == "f32" else 128
        rows = unit * max(1, _log(rng, 128, 8192) // unit)
        cols = 64 * max(1, min(_log(rng, 64, VOCAB), HIDDEN * VOCAB // rows) // 64)
        return {"kind": kind, "rows": rows, "cols": cols, "fmt": fmt}
    if kind == "native":
        t = rng.choice(sorted(_NATIVE))
        unit = 256 if t in ("Q4_K", "Q6_K") else 32
        cols = unit * max(1, _log(rng, 256, 8192) // unit)
        rows = min(_log(rng, 64, VOCAB), HIDDEN * VOCAB // 2 // cols)
        return {"kind": kind, "type": t, "rows": rows, "cols": cols}
    if kind == "decode_layer":
        return {"kind": kind, "ctx": _log(rng, 2, 8191), "window": rng.choice([0, 0, 512]), "fmt": fmt}
    if kind == "prefill_attention":
        tokens = _log(rng, 2, 1024)
        return {"kind": kind, "tokens": tokens, "start": rng.choice([0, 0, _log(rng, 1, 1024)]),
                "window": rng.choice([0, 512])}
    if kind == "sample":
        k = rng.choice([0, 1, 20, 40, 64])
        return {"kind": kind, "vocab": _log(rng, 4096, VOCAB), "k": k,
                "parts": rng.choice([256, 256, 1024] if k else [256, 1024, 4096])}
    layers = rng.choice([1, 2, 6, 6, 26])
    if kind == "prefill":
        tokens = _log(rng, 3, 2000)
        return {"kind": kind, "layers": layers, "tokens": tokens, "start": rng.choice([0, 0, _log(rng, 1, 1500)]),
                "fmt": fmt}
    if kind == "decode":
        return {"kind": kind, "layers": layers, "ctx": _log(rng, 1, 8000), "steps": rng.randint(1, 16), "fmt": fmt}
    return {"kind": "batch", "layers": layers, "seqs": rng.choice([1, 2, 5, 8, 16]), "depth": _log(rng, 16, 4096),
            "steps": rng.randint(1, 8), "fmt": fmt}


# ---- inputs ----------------------------------------------------------------

def _gen(case, seed):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + len(str(sorted(case.items()))))


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std


def _words(g, nbytes):
    return torch.randint(0, 256, (nbytes,), generator=g, device=DEV, dtype=torch.uint8)


def _int4(g, rows, cols, fmt):
    """A KM4 nibble plane and its scale plane (the planes' orders are in include/xpose.h)."""
    wq = _words(g, rows * cols // 2)
    sc = _normal(g, rows // 32 * cols, std=0.02).abs()
    return wq, sc.to({"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[fmt])


def _dequant(wq, sc, rows, cols):
    """[rows][cols] in float64 of a KM4 plane: uint4 (g, b, t) = columns 64 g + t, rows 32 b ..."""
    nblk = rows // 32
    w = wq.view(cols // 64, nblk, 64, 16)                       # byte i of a block: rows 2 i, 2 i + 1
    n = torch.stack((w & 15, w >> 4), -1).reshape(cols // 64, nblk, 64, 32).to(F64) - 8
    s = sc.view(nblk, cols) if sc.dtype == torch.float32 else \
        sc.view(nblk // 4, cols, 4).permute(0, 2, 1).reshape(nblk, cols)
    s = s.to(F64).view(nblk, cols // 64, 64).permute(1, 0, 2)
    return (n * s[..., None]).permute(1, 3, 0, 2).reshape(rows, cols)


_NATIVE = {"Q5_0": X.GGML_Q5_0, "Q8_0": X.GGML_Q8_0, "Q4_K": X.GGML_Q4_K, "Q6_K": X.GGML_Q6_K}


def _native_planes(g, c):
    """Repacked planes of a native-format matrix (xp_rq_tensor in include/xpose.h)."""
    slots = -(-c["rows"] // 64) * (c["cols"] // 32) * 64
    t = c["type"]
    return {"quant": _words(g, slots * (32 if t == "Q8_0" else 16)),
            "high": _words(g, slots * (4 if t == "Q5_0" else 8)) if t in ("Q5_0", "Q6_K") else None,
            "scale": _normal(g, slots * (2 if t == "Q6_K" else 1), std=0.02 if t != "Q8_0" else 0.002).abs(),
            "bias": _normal(g, slots, std=0.1).abs() if t == "Q4_K" else None}


def _native_dequant(p, c):
    t, nkb, n = c["type"], c["cols"] // 32, -(-c["rows"] // 64)
    if t == "Q8_0":
        q = p["quant"].view(torch.int8).view(-1, 32).to(F64)
    else:
        b = p["quant"].view(-1, 16)
        q = torch.stack((b & 15, b >> 4), -1).view(-1, 32).to(torch.int32)
        if t == "Q5_0":
            h = p["high"].view(-1, 4, 1).to(torch.int32) >> torch.arange(8, device=DEV, dtype=torch.int32)
            q = q + 16 * (h & 1).reshape(-1, 32) - 16
        elif t == "Q6_K":
            h = p["high"].view(-1, 8, 1).to(torch.int32) >> torch.arange(0, 8, 2, device=DEV, dtype=torch.int32)
            q = q + 16 * (h & 3).reshape(-1, 32) - 32
        q = q.to(F64)
    s = p["scale"].to(F64)
    s = s.view(-1, 2).repeat_interleave(16, 1) if t == "Q6_K" else s.view(-1, 1)
    w = q * s
    if p["bias"] is not None:
        w = w - p["bias"].to(F64).view(-1, 1)
    return w.view(n, nkb, 64, 32).permute(0, 2, 1, 3).reshape(n * 64, c["cols"])[:c["rows"]]


MATS = {X.T_Q: (HIDDEN, HEADS * HD), X.T_K: (HIDDEN, HD), X.T_V: (HIDDEN, HD), X.T_O: (HEADS * HD, HIDDEN),
        X.T_GATE: (HIDDEN, FFN), X.T_UP: (HIDDEN, FFN), X.T_DOWN: (FFN, HIDDEN)}


def _layer_weights(g, fmt):
    w = {m: _int4(g, *MATS[m], fmt) for m in MATS}
    w.update({n: _normal(g, HD if n >= X.T_Q_NORM else HIDDEN, std=0.1) for n in X.NORMS})
    return w


def _is_global(layer):
    return (layer + 1) % 6 == 0


def _model(c, seed, max_seq):
    """A session on a model of c["layers"] layers, and (keep) its weights for exact()."""
    g = _gen(c, seed)
    layers = [_layer_weights(g, c["fmt"]) for _ in range(c["layers"])]
    head = _int4(g, HIDDEN, VOCAB, c["fmt"])
    final = _normal(g, HIDDEN, std=0.1)
    return g, layers, head, final


def _host(t):
    return t.cpu().view(torch.uint8).numpy()


def _session(c, model, max_seq):
    _, layers, head, final = model
    sess = X.DecodeSession(X.XpConfig.gemma3_1b(n_layers=c["layers"], max_seq=max_seq, scale_fmt=FMT[c["fmt"]]))
    for l, w in enumerate(layers):
        for m in MATS:
            sess.upload(l, m, _host(w[m][0]))
            sess.upload(l, m | X.T_SCALES, _host(w[m][1]))
        for n in X.NORMS:
            sess.upload(l, n, _host(w[n]))
    sess.upload(-1, X.T_LM_HEAD, _host(head[0]))
    sess.upload(-1, X.T_LM_HEAD | X.T_SCALES, _host(head[1]))
    sess.upload(-1, X.T_FINAL_NORM, _host(final))
    return sess


def _max_seq(c):
    need = {"prefill": c.get("start", 0) + c.get("tokens", 0), "decode": c.get("ctx", 0) + c.get("steps", 0) + 1,
            "batch": c.get("depth", 0) + c.get("steps", 0) + 1}[c["kind"]]
    return min(8192, -(-need // 1024) * 1024)


def _kv(g, rows):
    return torch.randn(2, rows, HD, generator=g, device=DEV, dtype=torch.float32).half()


def _depths(c):
    """The sequences' positions: spread from a sixteenth of the deepest to it."""
    n = c["seqs"]
    return [max(1, c["depth"] * (i + 1) // n) for i in range(n)]


_ready = False


def _engine_inputs(c, seed):
    """The model, the token ids and the KV rows that an engine-level case starts from."""
    model = _model(c, seed, _max_seq(c))
    g = model[0]
    kind = c["kind"]
    n_ids = {"prefill": c.get("tokens"), "decode": 1, "batch": c.get("seqs")}[kind]
    ids = torch.randint(0, VOCAB, (n_ids,), generator=g, device=DEV).cpu().numpy().astype(np.uint32)
    rows = {"prefill": [c.get("start", 0)], "decode": [c.get("ctx", 0)]}.get(kind) or _depths(c)
    kv = [[_kv(g, r) for r in rows] for _ in range(c["layers"])]
    return model, ids, rows, kv


def prepare(case, seed):
    global _ready
    if not _ready:
        X.init(0)
        _ready = True
    c, kind = case, case["kind"]
    if kind in ("prefill", "decode", "batch"):
        model, ids, rows, kv = _engine_inputs(c, seed)
        sess = _session(c, model, _max_seq(c))
        st = {"case": c, "sess": sess, "ids": ids, "rows": rows}
        if kind == "batch":
            st["batch"] = X.DecodeBatch(sess, c["seqs"], _max_seq(c))
            put = st["batch"].kv_upload
        else:
            def put(_, *a):
                return sess.kv_upload(*a)
        for l, per in enumerate(kv):
            for s, t in enumerate(per):
                if t.shape[1]:
                    h = t.view(torch.int16).cpu().numpy().view(np.uint16)
                    put(s, l, 0, 0, h[0])
                    put(s, l, 1, 0, h[1])
        return st
    g = _gen(c, seed)
    st = {"case": c}
    if kind == "matvec":
        st["w"], st["s"] = _int4(g, c["rows"], c["cols"], c["fmt"])
        st["x"] = _normal(g, c["rows"])
        st["y"] = torch.empty(c["cols"], device=DEV)
    elif kind == "native":
        st["p"] = p = _native_planes(g, c)
        st["x"] = _normal(g, c["cols"])
        st["y"] = torch.empty(c["rows"], device=DEV)
        t = X.RqTensor()
        t.type, t.rows, t.cols = _NATIVE[c["type"]], c["rows"], c["cols"]
        for k, v in p.items():
            setattr(t, k, v.data_ptr() if v is not None else None)
        st["t"] = t
    elif kind == "decode_layer":
        st["w"] = _layer_weights(g, c["fmt"])
        st["x0"] = _normal(g, HIDDEN, std=4.0)
        st["k"], st["v"] = _kv(g, c["ctx"]).unbind(0)
        f = {n: torch.empty(k, device=DEV) for n, k in dict(
            x=HIDDEN, h=HIDDEN, q=HEADS * HD, kr=HD, vr=HD, qo=HEADS * HD, ko=HD, att=HEADS * HD, o=HIDDEN,
            gate=FFN, up=FFN, act=FFN).items()}
        st.update(f)
    elif kind == "prefill_attention":
        t, s = c["tokens"], c["start"] + c["tokens"]
        st["q_raw"], st["k_raw"], st["v_raw"] = _normal(g, t, HEADS, HD), _normal(g, t, 1, HD), _normal(g, t, HD)
        st["qw"], st["kw"] = _normal(g, HD, std=0.1), _normal(g, HD, std=0.1)
        st["kc"], st["vc"] = _normal(g, s, HD), _normal(g, s, HD)
        f = dict(q=(t, HEADS, HD), k=(t, 1, HD), scores=(HEADS, t, s), stats=(HEADS * t, 2), out=(HEADS, t, HD))
        st.update({n: torch.empty(*v, device=DEV) for n, v in f.items()})
    elif kind == "sample":
        n, k, p = c["vocab"], c["k"], c["parts"]
        st["logits"] = _normal(g, (n + 3) // 4 * 4, std=3.0)
        st["u"] = float(torch.rand(1, generator=g, device=DEV))
        f = dict(x=st["logits"].numel(), pmax=p, psum=p, stats=2, cval=max(1, p * k), oval=64, w=64, out=2)
        st.update({a: torch.empty(b, device=DEV) for a, b in f.items()})
        st.update({a: torch.empty(b, device=DEV, dtype=torch.int32) for a, b in
                   dict(cidx=max(1, p * k), oidx=64, tok=1).items()})
    return st


# ---- one pass --------------------------------------------------------------

def _p(t):
    return t.data_ptr()


def _run_decode_layer(st):
    c, w, fmt = st["case"], st["w"], FMT[st["case"]["fmt"]]
    call = X.call
    x, h, pos = _p(st["x"]), _p(st["h"]), c["ctx"] - 1
    theta = C.c_float(THETA[c["window"] == 0])

    def multi(mats, outs, src):
        n = len(mats)
        call("xp_mv_int4_multi", n, (C.c_void_p * n)(*outs), src, (C.c_void_p * n)(*[_p(w[m][0]) for m in mats]),
             (C.c_void_p * n)(*[_p(w[m][1]) for m in mats]), (C.c_uint32 * n)(*[MATS[m][1] for m in mats]), fmt,
             MATS[mats[0]][0], None)

    def one(m, out, src):
        call("xp_mv_int4", out, src, _p(w[m][0]), _p(w[m][1]), fmt, MATS[m][0], MATS[m][1], 0, None)

    def norm(out, src, n):
        call("xp_rmsnorm_gemma", out, src, _p(w[n]), HIDDEN, EPS, None)

    q, kr, vr, qo, ko, att, o, gate, up, act = (_p(st[n]) for n in (
        "q", "kr", "vr", "qo", "ko", "att", "o", "gate", "up", "act"))
    call("xp_copy", x, _p(st["x0"]), HIDDEN * 4, None)
    norm(h, x, X.T_ATTN_NORM)
    multi((X.T_Q, X.T_K, X.T_V), (q, kr, vr), h)
    call("xp_qk_norm_rope_append", qo, ko, q, kr, vr, _p(w[X.T_Q_NORM]), _p(w[X.T_K_NORM]), _p(st["k"]),
         _p(st["v"]), HEADS, 1, HD, pos, theta, EPS, None)
    span = min(c["ctx"], c["window"]) if c["window"] else c["ctx"]
    call("xp_attention_decode", att, qo, _p(st["k"]), _p(st["v"]), HEADS, 1, HD, span, c["ctx"] - span, 1 / 16, None)
    one(X.T_O, o, att)
    norm(o, o, X.T_POST_ATTN_NORM)
    call("xp_add_residual", x, o, HIDDEN, None)
    norm(h, x, X.T_FFN_NORM)
    multi((X.T_GATE, X.T_UP), (gate, up), h)
    call("xp_geglu", act, gate, up, FFN, None)
    one(X.T_DOWN, o, act)
    norm(o, o, X.T_POST_FFN_NORM)
    call("xp_add_residual", x, o, HIDDEN, None)
    return {n: st[n] for n in ("x", "att", "act", "qo", "k", "v")}


def _run_prefill_attention(st):
    c, call = st["case"], X.call
    t, s, pos0 = c["tokens"], c["start"] + c["tokens"], c["start"]
    theta = C.c_float(THETA[c["window"] == 0])
    call("xp_rmsnorm_heads_rows_gemma", _p(st["q"]), _p(st["q_raw"]), _p(st["qw"]), t, HEADS, HD, EPS, None)
    call("xp_rmsnorm_heads_rows_gemma", _p(st["k"]), _p(st["k_raw"]), _p(st["kw"]), t, 1, HD, EPS, None)
    call("xp_rope_prefill", _p(st["q"]), t, HEADS, HD, pos0, theta, None)
    call("xp_rope_prefill", _p(st["k"]), t, 1, HD, pos0, theta, None)
    call("xp_kv_append_rows", _p(st["kc"]), _p(st["k"]), t, HD, pos0, None)
    call("xp_kv_append_rows", _p(st["vc"]), _p(st["v_raw"]), t, HD, pos0, None)
    q = st["q"].transpose(0, 1).contiguous()          # the scores take [head][query][dim]
    call("xp_attention_scores_prefill", _p(st["scores"]), _p(q), _p(st["kc"]), HEADS, 1, HD, t, s, pos0, c["window"],
         1 / 16, None)
    call("xp_softmax_rows_stats", _p(st["stats"]), _p(st["scores"]), HEADS * t, s, None)
    call("xp_softmax_rows_apply", _p(st["scores"]), _p(st["stats"]), HEADS * t, s, None)
    call("xp_attention_apply_prefill", _p(st["out"]), _p(st["scores"]), _p(st["vc"]), HEADS, 1, HD, t, s, None)
    return {"out": st["out"], "probs": st["scores"], "k": st["kc"], "v": st["vc"]}


def _run_sample(st):
    c, call = st["case"], X.call
    n, k, parts = c["vocab"], c["k"], c["parts"]
    x, stats, w, psum, out, tok = (_p(st[a]) for a in ("x", "stats", "w", "psum", "out", "tok"))
    call("xp_copy", x, _p(st["logits"]), st["x"].numel() * 4, None)
    call("xp_apply_temperature", x, 1 / 0.8, n, None)
    if k == 0:
        call("xp_reduce_max_partial", _p(st["pmax"]), x, n, parts, None)
        call("xp_reduce_max_final", stats, _p(st["pmax"]), parts, None)
        call("xp_softmax_exp_partial", x, psum, x, stats, n, parts, None)
        call("xp_reduce_sum_final", stats, psum, parts, None)
        call("xp_multinomial_strided", out, tok, x, psum, stats, n, parts, st["u"], None)
        call("xp_softmax_normalize", x, stats, n, None)
        return {"probs": st["x"][:n], "token": st["tok"], "draw": st["out"]}
    call("xp_topk_partial", _p(st["cval"]), _p(st["cidx"]), x, n, parts, k, None)
    call("xp_topk_rank_select", _p(st["oval"]), _p(st["oidx"]), _p(st["cval"]), _p(st["cidx"]), parts * k, k, None)
    call("xp_reduce_max_final", stats, _p(st["oval"]), k, None)
    call("xp_softmax_exp_partial", w, psum, _p(st["oval"]), stats, k, k, None)
    call("xp_topp_cutoff", w, k, 0.95, None)
    call("xp_multinomial_sample", out, tok, w, _p(st["oidx"]), k, st["u"], None)
    return {"values": st["oval"][:k], "ids": st["oidx"][:k], "weights": st["w"][:k], "token": st["tok"],
            "cval": st["cval"], "cidx": st["cidx"]}


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "matvec":
        X.call("xp_mv_int4", _p(st["y"]), _p(st["x"]), _p(st["w"]), _p(st["s"]), FMT[c["fmt"]], c["rows"], c["cols"],
               0, None)
        return st["y"]
    if kind == "native":
        X.call("xp_mv_rq", _p(st["y"]), _p(st["x"]), C.byref(st["t"]), 0, None)
        return st["y"]
    if kind == "decode_layer":
        return _run_decode_layer(st)
    if kind == "prefill_attention":
        return _run_prefill_attention(st)
    if kind == "sample":
        return _run_sample(st)
    sess = st["sess"]
    if kind == "prefill":
        sess.set_position(c["start"])
        sess.prefill(st["ids"])
        # the last layer's KV rows depend on every row of every layer before
        last = c["layers"] - 1
        kv = [sess.kv_download(last, w, c["start"], c["tokens"]).view(np.float16) for w in (0, 1)]
        return {"logits": sess.last_logits(), "k": kv[0], "v": kv[1]}
    if kind == "decode":
        sess.set_position(c["ctx"])
        sess.prefill(st["ids"])
        tokens = sess.decode_steps(c["steps"])
        return {"tokens": tokens.astype(np.int64), "logits": sess.last_logits()}
    b = st["batch"]
    b.set_positions(st["rows"])
    b.forward(st["ids"])
    tokens = b.decode_steps(c["steps"])
    return {"tokens": tokens.astype(np.int64), "logits": [b.last_logits(i) for i in range(c["seqs"])]}


# ---- the work a pass cannot do without -------------------------------------

def _int4_bytes(rows, cols, fmt):
    return rows * cols / 2 + rows // 32 * cols * (4 if fmt == "f32" else 2)


_LAYER_WEIGHTS = sum(r * k for r, k in MATS.values())


def _attended(start, tokens, window):
    """Key positions that queries start .. start + tokens - 1 attend to, added up."""
    return sum(min(p + 1, window) if window else p + 1 for p in range(start, start + tokens))


def work(case):
    c, kind = case, case["kind"]
    if kind == "matvec":
        return {"bytes": _int4_bytes(c["rows"], c["cols"], c["fmt"]) + 4 * (c["rows"] + c["cols"]),
                "flops": 2 * c["rows"] * c["cols"]}
    if kind == "native":
        per = {"Q8_0": 36, "Q5_0": 24, "Q4_K": 24, "Q6_K": 32}[c["type"]]
        return {"bytes": c["rows"] * c["cols"] // 32 * per + 4 * (c["rows"] + c["cols"]),
                "flops": 2 * c["rows"] * c["cols"]}
    if kind == "decode_layer":
        span = min(c["ctx"], c["window"]) if c["window"] else c["ctx"]
        return {"bytes": sum(_int4_bytes(r, k, c["fmt"]) for r, k in MATS.values()) + span * 1024 + 8 * HIDDEN,
                "flops": 2 * _LAYER_WEIGHTS + span * HEADS * HD * 4}
    if kind == "prefill_attention":
        t, s = c["tokens"], c["start"] + c["tokens"]
        # q, k, v in; the cache's earlier rows; k, v, the probabilities and the output
        return {"bytes": 4 * (t * (HEADS + 2) * HD + 2 * c["start"] * HD + 2 * t * HD + HEADS * t * s + HEADS * t * HD),
                "flops": 4 * HEADS * HD * _attended(c["start"], t, c["window"])}
    if kind == "sample":
        n = c["vocab"]
        return {"bytes": 4 * n * 2 if c["k"] == 0 else 4 * n + 8 * c["parts"] * c["k"], "flops": 4 * n}
    head = _int4_bytes(HIDDEN, VOCAB, c["fmt"]) + 4 * VOCAB
    layer = sum(_int4_bytes(r, k, c["fmt"]) for r, k in MATS.values())
    L = c["layers"]
    wins = [0 if _is_global(l) else 512 for l in range(L)]
    if kind == "prefill":
        t, s0 = c["tokens"], c["start"]
        kv = sum((t + (min(s0, w) if w else s0)) * 1024 for w in wins)
        att = sum(_attended(s0, t, w) for w in wins)
        return {"bytes": L * layer + head + kv, "flops": 2 * t * L * _LAYER_WEIGHTS + 2 * HIDDEN * VOCAB
                + 4 * HEADS * HD * att}
    steps = c["steps"] + 1
    at = [c["ctx"]] if kind == "decode" else _depths(c)
    keys = sum(_attended(p, steps, w) for p in at for w in wins)
    return {"bytes": steps * (L * layer + head + 4 * VOCAB * (len(at) - 1)) + 1024 * keys,
            "flops": steps * len(at) * 2 * (L * _LAYER_WEIGHTS + HIDDEN * VOCAB) + 4 * HEADS * HD * keys}


def tolerance(case):
    # about four times the distance from float64: 20-bit block fixed point in
    # the matvecs (2.6e-6), float32 sums elsewhere; in a whole model the
    # float16 rounding of a cache row falls to the other side now and then,
    # which a short context shows most (2.5e-5 to 4e-5; "max": a float16 step
    # is up to 2^-10 of a value)
    kind = case["kind"]
    if kind in ("matvec", "native"):
        return {"rel": 1e-5}
    if kind == "sample":
        return {"rel": 5e-6}
    if kind == "decode_layer":
        return {"rel": 1e-4, "max": 4e-3}
    if kind == "prefill_attention":
        return {"rel": 2e-6}
    return {"rel": 1.5e-4, "max": 4e-3}


# ---- float64 ---------------------------------------------------------------

def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (1 + w.to(F64))


def _rope64(x, pos, theta):
    """x [..., rows, heads, HD] rotated at positions pos [rows]; the angle is a product of two float32 values,
    as the entry points define it."""
    d = torch.arange(HD // 2, dtype=torch.float32)
    inv = torch.exp2((-torch.log2(torch.tensor(theta)) * (2 * d / HD)).to(F64)).to(torch.float32)
    ang = (pos.to(torch.float32)[:, None] * inv.to(DEV)).to(F64)[:, None, :]
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()), -1)


def _attend64(q, k, v, pos, window):
    """q [t, HEADS, HD] at positions pos over rows k, v [s, HD]: out [t, HEADS, HD], probabilities [HEADS, t, s]."""
    s = torch.matmul(q.transpose(0, 1).reshape(-1, HD), k.t().contiguous()).view(HEADS, q.shape[0], -1) / 16
    t = torch.arange(k.shape[0], device=DEV)[None]
    off = t > pos[:, None]
    if window:
        off |= t + window <= pos[:, None]
    p = s.masked_fill_(off, -math.inf).softmax(-1)
    o = torch.matmul(p.reshape(-1, k.shape[0]), v).view(HEADS, q.shape[0], HD).transpose(0, 1)
    return o, p


def _layer64(x, w, kc, vc, pos, window):
    """One layer on rows x [t, HIDDEN] at positions pos; kc, vc [start, HD] are the rows before. Also the layer's
    cache rows (float16, as the cache holds them), its attention output, activation and queries."""
    W = {m: w[m] if torch.is_tensor(w[m]) else _dequant(*w[m], *MATS[m]) for m in MATS}
    h = _norm64(x, w[X.T_ATTN_NORM])
    theta = THETA[window == 0]
    q = _rope64(_norm64((h @ W[X.T_Q]).view(-1, HEADS, HD), w[X.T_Q_NORM]), pos, theta)
    k = _rope64(_norm64((h @ W[X.T_K]).view(-1, 1, HD), w[X.T_K_NORM]), pos, theta)[:, 0]
    k, v = torch.cat((kc, k.half())), torch.cat((vc, (h @ W[X.T_V]).half()))
    att, _ = _attend64(q, k.to(F64), v.to(F64), pos, window)
    att = att.reshape(-1, HEADS * HD)
    x = x + _norm64(att @ W[X.T_O], w[X.T_POST_ATTN_NORM])
    h = _norm64(x, w[X.T_FFN_NORM])
    act = torch.nn.functional.gelu(h @ W[X.T_GATE], approximate="tanh") * (h @ W[X.T_UP])
    x = x + _norm64(act @ W[X.T_DOWN], w[X.T_POST_FFN_NORM])
    return x, k, v, att, act, q


def _engine64(c, seed):
    (_, layers, head, final), ids, rows, kv = _engine_inputs(c, seed)
    head = _dequant(*head, HIDDEN, VOCAB)
    layers = [{n: _dequant(*t, *MATS[n]) if n in MATS else t for n, t in w.items()} for w in layers]
    steps = c.get("steps", 0)
    tokens = np.zeros((steps, len(rows)), np.int64)
    logits = []
    for s, start in enumerate(rows):
        cache = [list(per[s].unbind(0)) for per in kv]
        now = [int(i) for i in (ids if c["kind"] == "prefill" else ids[s:s + 1])]
        for step in range(steps + 1):
            x = head[:, now].t() * float(np.float32(math.sqrt(HIDDEN)))
            pos = torch.arange(start, start + len(now), device=DEV)
            start += len(now)
            for l, w in enumerate(layers):
                x, cache[l][0], cache[l][1] = _layer64(x, w, *cache[l], pos, 0 if _is_global(l) else 512)[:3]
            out = _norm64(x[-1], final) @ head
            if step < steps:
                now = [int(out.argmax())]
                tokens[step, s] = now[0]
        logits.append(out)
    if c["kind"] == "prefill":
        k, v = (t[c["start"]:].reshape(-1) for t in cache[-1])
        return {"logits": logits[0], "k": k, "v": v}
    if c["kind"] == "decode":
        return {"tokens": tokens[:, 0], "logits": logits[0]}
    return {"tokens": tokens, "logits": logits}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("prefill", "decode", "batch"):
        return _engine64(c, seed)
    g = _gen(c, seed)
    if kind == "matvec":
        w = _int4(g, c["rows"], c["cols"], c["fmt"])
        return _normal(g, c["rows"]).to(F64) @ _dequant(*w, c["rows"], c["cols"])
    if kind == "native":
        p = _native_planes(g, c)
        return _native_dequant(p, c) @ _normal(g, c["cols"]).to(F64)
    st = prepare(c, seed)
    if kind == "decode_layer":
        n = c["ctx"] - 1
        x, k, v, att, act, q = _layer64(st["x0"].to(F64)[None], st["w"], st["k"][:n], st["v"][:n],
                                        torch.tensor([n], device=DEV), c["window"])
        return {"x": x[0], "att": att[0], "act": act[0], "qo": q.reshape(-1), "k": k, "v": v}
    if kind == "prefill_attention":
        s0 = c["start"]
        pos = torch.arange(s0, s0 + c["tokens"], device=DEV)
        theta = THETA[c["window"] == 0]
        q = _rope64(_norm64(st["q_raw"].to(F64), st["qw"]), pos, theta)
        k = _rope64(_norm64(st["k_raw"].to(F64), st["kw"]), pos, theta)[:, 0]
        k = torch.cat((st["kc"][:s0].to(F64), k))
        v = torch.cat((st["vc"][:s0], st["v_raw"])).to(F64)
        o, p = _attend64(q, k, v, pos, c["window"])
        return {"out": o.transpose(0, 1).contiguous(), "probs": p, "k": k, "v": v}
    x = st["logits"][:c["vocab"]].to(F64) / 0.8
    if c["k"] == 0:
        return {"probs": x.softmax(0), "token": None, "draw": None}
    top = x.topk(c["k"]).values
    return {"values": top, "ids": None, "weights": None, "token": None, "cval": None, "cidx": None}
