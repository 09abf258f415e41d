"""Prompt prefill through the GEMM engine (xp_session_prefill, XP_PREFILL_AUTO,
prompts of more than 17 tokens, and shorter ones of shapes that the batched step
does not take) against XP_PREFILL_TOKENS, the token steps that
tests/test_session.py holds to the oracle: every KV row the prompt appends, in
layers below a local and a global attention, and the last logits.

Tolerance: one float16 step of a row's largest value (2^-10, 1e-3), and of all
rows together 2e-4 in the 2-norm. Activations are two bf16 terms, so before it
is rounded a cache value differs by d = 2^-18 to 2^-16 of itself, and rounds to
the other side of a 2^-11 step with probability d / 2^-11: sqrt(2^-11 d) = 4e-5 to
9e-5 (3.5e-5 to 7.6e-5 seen). The logits, which average over many such rows,
2e-5 (0.1e-6 to 4.2e-6 seen). Sizes are the edges of the engine's shapes: 32-, 64- and 128-row
workgroups with one row more and one less, prompts that end in a partly filled
tile, one that takes two chunks, spans split over workgroups, one to four
query heads a KV head, the sliding window's edge, both scale formats."""
import ctypes as C
import os

import numpy as np
import pytest

SHAPES = {"gemma": dict(hidden=1152, ffn=6912, n_heads=4, n_kv_heads=1),
          "narrow": dict(hidden=512, ffn=1024, n_heads=2, n_kv_heads=1),
          "mha": dict(hidden=384, ffn=640, n_heads=2, n_kv_heads=2),
          "wide": dict(hidden=2048, ffn=1152, n_heads=4, n_kv_heads=2),
          "split": dict(hidden=2048, ffn=8192, n_heads=4, n_kv_heads=2),   # no batched step for it
          "h2176": dict(hidden=2176, ffn=384, n_heads=2, n_kv_heads=1), "h4096": dict(hidden=4096, ffn=384, n_heads=2, n_kv_heads=1),
          "h4224": dict(hidden=4224, ffn=384, n_heads=2, n_kv_heads=1), "h8192": dict(hidden=8192, ffn=256, n_heads=2, n_kv_heads=1)}


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tokens,start,fmt", [
    ("gemma", 18, 0, "f16"), ("gemma", 33, 700, "bf16"), ("gemma", 34, 3, "f16"), ("gemma", 65, 0, "bf16"),
    ("gemma", 66, 500, "f16"), ("gemma", 129, 0, "f16"), ("gemma", 130, 1001, "bf16"), ("gemma", 300, 333, "f16"),
    ("gemma", 40, 3000, "f16"), ("narrow", 47, 5, "f16"), ("narrow", 258, 0, "bf16"), ("narrow", 2100, 0, "f16"),
    ("mha", 31, 600, "f16"), ("mha", 161, 0, "f16"), ("wide", 20, 90, "f16"), ("wide", 200, 450, "bf16"),
    ("split", 3, 0, "f16"), ("split", 17, 30, "bf16"), ("split", 40, 5, "f16"),
    ("h2176", 70, 0, "f16"), ("h4096", 130, 0, "f16"), ("h4224", 20, 7, "f16"), ("h8192", 90, 0, "f16"),
    ("gemma", 513, 0, "f16"), ("gemma", 514, 0, "f16")])
def test_gpu_prefill_engine_equals_token_steps(xp, shape, tokens, start, fmt):
    X = xp
    print(f"case prefill engine {shape} tokens={tokens} start={start} {fmt}", flush=True)
    sf = {"f16": X.XP_SCALE_F16_QUAD, "bf16": X.XP_SCALE_BF16_QUAD}[fmt]
    got = []
    for pm in (X.XP_PREFILL_AUTO, X.XP_PREFILL_TOKENS):
        # layer 0 local, layer 1 global, layer 2's KV rows depend on both
        cfg = X.XpConfig.gemma3_1b(n_layers=3, vocab=1024, global_every=2, max_seq=max(512, start + tokens),
                                   scale_fmt=X.XP_SCALE_F16_QUAD, prefill_mode=pm, **SHAPES[shape])
        kvd = cfg.n_kv_heads * cfg.head_dim
        rng = np.random.default_rng(tokens)
        synth = {}
        for l in range(cfg.n_layers):
            for t in X.MATRICES + X.NORMS + tuple(m | X.T_SCALES for m in X.MATRICES):
                synth[l, t] = X.synth_tensor(cfg, 11, l, t)
        for t in (X.T_LM_HEAD, X.T_LM_HEAD | X.T_SCALES, X.T_FINAL_NORM):
            synth[-1, t] = X.synth_tensor(cfg, 11, -1, t)
        cfg.scale_fmt = sf
        sess = X.DecodeSession(cfg)
        for (l, t), a in synth.items():
            if t & X.T_SCALES and fmt == "bf16":
                f = a.view(np.float16).astype(np.float32)
                a = (f.view(np.uint32) >> 16).astype(np.uint16)
            sess.upload(l, t, a)
        for l in range(cfg.n_layers):
            for which in (0, 1):
                if start:
                    sess.kv_upload(l, which, 0, X.synth_normal_f16(start * kvd, 5, 2 * l + which))
        sess.set_position(start)
        sess.prefill(rng.integers(0, cfg.vocab, tokens).astype(np.uint32))
        assert sess.position == start + tokens
        rows = [sess.kv_download(l, w, start, tokens).view(np.float16).astype(np.float64).reshape(tokens, kvd)
                for l in range(cfg.n_layers) for w in (0, 1)]
        got.append((rows, sess.last_logits().astype(np.float64)))
        sess.close()
    (a, la), (b, lb) = got
    for i, (x, y) in enumerate(zip(a, b)):
        err = np.abs(x - y).max(axis=1)
        assert np.all(err <= 1e-3 * np.abs(y).max(axis=1)), (i, int(err.argmax()), err.max())
        assert np.linalg.norm(x - y) <= 2e-4 * np.linalg.norm(y), i
    assert np.abs(la - lb).max() <= 2e-5 * np.abs(lb).max()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tokens,start,window,cached,ahead", [
    # rows the workgroup's later rows no longer see, near and far ends of its 32 positions
    ("gemma", 40, 700, 512, (189, 195), ()), ("mha", 65, 600, 512, (90, 119), ()),
    ("narrow", 33, 40, 20, (25, 38), ()), ("mha", 40, 40, 1, (39,), ()),
    # rows ahead: the last of a tile of positions, the first of one, the keys of a split span
    ("gemma", 40, 0, 512, (), (7, 30)), ("mha", 130, 0, 512, (), (31, 128)), ("narrow", 70, 3000, 0, (), (17, 64)),
    ("gemma", 200, 3000, 0, (), (60, 197)), ("mha", 40, 40, 1, (39,), (20,))])
def test_gpu_prefill_engine_non_finite_values(xp, shape, tokens, start, window, cached, ahead):
    """A value row that is not finite reaches the positions that see it and no
    other: rows already cached that leave a window inside the prompt, and rows
    of the prompt itself whose values pass float16's largest, ahead of others.
    Layer 1's KV rows show layer 0's attention: XP_PREFILL_TOKENS (a token step
    reads its own span only) gives those of the positions that see none."""
    X = xp
    print(f"case prefill engine not finite {shape} tokens={tokens} start={start} window={window}", flush=True)
    bad_tok = 5
    got = {}
    for pm in (X.XP_PREFILL_AUTO, X.XP_PREFILL_TOKENS):
        cfg = X.XpConfig.gemma3_1b(n_layers=2, vocab=1024, global_every=2 if window else 0, max_seq=max(512, start + tokens),
                                   sliding_window=window or 512, prefill_mode=pm, **SHAPES[shape])
        kvd = cfg.n_kv_heads * cfg.head_dim
        sess = X.DecodeSession(cfg)
        sess.synthesize(3)
        emb = np.random.default_rng(7).normal(0, 1, (cfg.vocab, cfg.hidden)).astype(np.float32)
        emb[bad_tok] = 0.0
        emb[bad_tok, 0] = 1.0                # its normed row: sqrt(hidden) in one place
        sess.upload(-1, X.T_EMBED, emb)
        if ahead:
            # that place's weight block scaled so that its nibbles of -8 overflow
            # (8 s sqrt(hidden) = 72 000), other tokens' values (32 nibbles of
            # about 4.6 s) far from it
            sc = X.synth_tensor(cfg, 3, 0, X.T_V | X.T_SCALES).view(np.float16).copy()
            sc[:4 * kvd:4] = 9000.0 / np.sqrt(cfg.hidden)
            sess.upload(0, X.T_V | X.T_SCALES, sc)
            sess.upload(0, X.T_ATTN_NORM, np.zeros(cfg.hidden, np.float32))
        for l in range(2):
            for which in (0, 1):
                if start:
                    rows = X.synth_normal_f16(start * kvd, 5, 2 * l + which).reshape(start, kvd)
                    for i, p in enumerate(cached):
                        if l == 0 and which == 1:
                            rows[p, i::16] = np.float16([np.inf, np.nan][i % 2]).view(np.uint16)
                    sess.kv_upload(l, which, 0, rows)
        sess.set_position(start)
        ids = np.random.default_rng(tokens).integers(6, cfg.vocab, tokens).astype(np.uint32)
        ids[list(ahead)] = bad_tok
        sess.prefill(ids)
        v0 = sess.kv_download(0, 1, start, tokens).view(np.float16).reshape(tokens, kvd)
        got[pm] = [sess.kv_download(1, w, start, tokens).view(np.float16).astype(np.float64).reshape(tokens, kvd) for w in (0, 1)]
        sess.close()
        bad = np.array(sorted(set(cached) | {start + i for i in np.flatnonzero(~np.isfinite(v0).all(1))}))
        assert set(bad) == set(cached) | {start + i for i in ahead}
    pos = np.arange(start, start + tokens)[:, None]
    sees = ((bad <= pos) & ((bad + window > pos) if window else True)).any(1)
    assert not sees.all()
    for a, b in zip(got[X.XP_PREFILL_AUTO], got[X.XP_PREFILL_TOKENS]):
        assert np.isfinite(b[~sees]).all()
        assert np.array_equal(np.isfinite(a).all(1)[:-1], ~sees[:-1])   # the last token takes a token step
        err = np.abs(a[~sees] - b[~sees]).max(axis=1)
        assert np.all(err <= 1e-3 * np.abs(b[~sees]).max(axis=1)), (int(err.argmax()), err.max())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,start,window,qscale,splits", [
    (32, 0, 0, 1.0, 2), (200, 1000, 0, 1.0, 5), (200, 1000, 512, 1.0, 2), (500, 0, 512, 1.5, 2), (300, 1500, 0, 1.5, 4)])
def test_gpu_prefill_engine_attention_error(xp, rows, start, window, qscale, splits):
    """The engine's attention by itself, from the row records it writes before
    they are staged, against float64 of the same queries and cache: no further
    off than xp_attention_decode, the token steps' attention, is on the same
    rows. Both are measured here, so the bar needs no constant but 5 % for the
    rows drawn (float32 sums in another order; 0.93 to 1.01 of it measured)."""
    X = xp
    print(f"case prefill attention error rows={rows} start={start} window={window}", flush=True)
    lib = C.CDLL(os.path.join(os.path.dirname(__file__), "native", "prefill_attention.so"))
    rec, G, D, n = lib.test_prefill_attention_record(), 4, 256, start + rows
    r = np.random.default_rng(rows + start)
    k, v = (r.normal(0, 1, (n, D)).astype(np.float16) for _ in range(2))
    q = (r.normal(0, qscale, (rows, G, D))).astype(np.float32)
    e = 13 - np.floor(np.log2(np.abs(q).max(-1, keepdims=True)))
    qq = q * np.exp2(e).astype(np.float32)
    qh = qq.astype(np.float16)
    ql = (qq - qh.astype(np.float32)).astype(np.float16)
    wgs = -(-rows * G // 32)
    buf = {m: X.DeviceBuffer.from_array(a) for m, a in dict(qh=qh, ql=ql, qs=np.exp2(-e).astype(np.float32), k=k, v=v, q=q).items()}
    pad = -(-rows // 32) * 32
    part, a, asum, out = (X.DeviceBuffer(4 * m) for m in (wgs * splits * 32 * rec, pad * G * D, pad * G * D // 32, G * D))
    f = C.c_float
    rc = lib.test_prefill_attention(buf["qh"].vp, buf["ql"].vp, buf["qs"].vp, buf["k"].vp, buf["v"].vp, rows, 1, G, start,
                                    window, f(0.0625), a.vp, asum.vp, part.vp, splits)
    assert rc == 0
    X.synchronize()
    p = part.download(np.float32).astype(np.float64).reshape(wgs, splits, 32, rec)
    w = np.exp2(p[..., 0] - p[..., 0].max(1, keepdims=True))       # record: max (of score log2(e)), sum, 2 unused, row
    got = ((w[..., None] * p[..., 4:]).sum(1) / (w * p[..., 1]).sum(1)[..., None]).reshape(-1, G, D)[:rows]
    step = np.empty((rows, G, D), np.float32)
    for i in range(rows):
        span = min(start + i + 1, window) if window else start + i + 1
        X.call("xp_attention_decode", out.vp, C.c_void_p(buf["q"].ptr + 4 * i * G * D), buf["k"].vp, buf["v"].vp, G, 1, D, span,
               start + i + 1 - span, f(0.0625), None)
        X.synchronize()
        step[i] = out.download(np.float32).reshape(G, D)
    s = (q.reshape(-1, D).astype(np.float64) @ k.astype(np.float64).T / 16).reshape(rows, G, n)
    t, pos = np.arange(n)[None], np.arange(start, n)[:, None]
    off = (t > pos) | ((t + window <= pos) if window else False)
    s = np.where(off[:, None], -np.inf, s)
    s = np.exp(s - s.max(-1, keepdims=True))
    want = ((s / s.sum(-1, keepdims=True)).reshape(-1, n) @ v.astype(np.float64)).reshape(rows, G, D)
    err, bar = (np.linalg.norm(x - want) / np.linalg.norm(want) for x in (got, step))
    print(f"engine {err:.3e} step {bar:.3e}", flush=True)
    assert err <= 1.05 * bar
