"""Prompt prefill through the GEMM engine (xp_session_prefill, XP_PREFILL_AUTO,
prompts of more than 17 tokens) against XP_PREFILL_TOKENS, the token steps that
tests/test_session.py holds to the oracle: every KV row the prompt appends, in
layers below a local and a global attention, and the last logits.

Tolerance: 1e-3 of a row's largest value, the bar the batched prefill has
against the oracle (activations as two bf16 terms, 2^-18; cache rows fp16,
2^-11). Sizes are the edges of the engine's shapes: 32-, 64- and 128-row
workgroups with one row more and one less, prompts that end in a partly filled
tile, one that takes two chunks, spans split over workgroups, one to four
query heads a KV head, the sliding window's edge, both scale formats."""
import numpy as np
import pytest

SHAPES = {"gemma": dict(hidden=1152, ffn=6912, n_heads=4, n_kv_heads=1),
          "narrow": dict(hidden=512, ffn=1024, n_heads=2, n_kv_heads=1),
          "mha": dict(hidden=384, ffn=640, n_heads=2, n_kv_heads=2),
          "wide": dict(hidden=2048, ffn=1152, n_heads=4, n_kv_heads=2)}


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tokens,start,fmt", [
    ("gemma", 18, 0, "f16"), ("gemma", 33, 700, "bf16"), ("gemma", 34, 3, "f16"), ("gemma", 65, 0, "bf16"),
    ("gemma", 66, 500, "f16"), ("gemma", 129, 0, "f16"), ("gemma", 130, 1001, "bf16"), ("gemma", 300, 333, "f16"),
    ("gemma", 40, 3000, "f16"), ("narrow", 47, 5, "f16"), ("narrow", 258, 0, "bf16"), ("narrow", 2100, 0, "f16"),
    ("mha", 31, 600, "f16"), ("mha", 161, 0, "f16"), ("wide", 20, 90, "f16"), ("wide", 200, 450, "bf16")])
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
    assert np.abs(la - lb).max() <= 1e-3 * np.abs(lb).max()
