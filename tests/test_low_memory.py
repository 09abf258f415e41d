"""Refused device allocations: what they leave behind, and the prompt prefill's
way on from them (fewer positions a pass, the batched step, token steps). The
prefill cases run in a process of their own, where tests/native/alloc_limit.cpp
stands before the runtime's hipMalloc and has it refuse what is above a limit."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
def test_gpu_refused_allocation_is_reported_once(xp):
    """The call that failed says so; the next launch is not failed for it."""
    X = xp
    print("case refused allocation", flush=True)
    x = X.DeviceBuffer.from_array(np.arange(8, dtype=np.float32))
    with pytest.raises(X.XposeError) as e:
        X.DeviceBuffer(1 << 50)
    assert "hipMalloc" in str(e.value)
    X.call("xp_apply_temperature", x.vp, 0.5, 8, None)
    X.synchronize()
    assert np.array_equal(x.download(np.float32), np.arange(8, dtype=np.float32) / 2)


class Child:
    """A session's prompts under a limit, against XP_PREFILL_TOKENS without one."""

    def __init__(self):
        self.lim = C.CDLL(os.path.join(ROOT, "tests", "native", "alloc_limit.so"), mode=C.RTLD_GLOBAL)
        sys.path.insert(0, ROOT)
        import xpose_amd
        self.X = xpose_amd
        self.X.init(0)

    def var(self, name, t=C.c_size_t):
        return t.in_dll(self.lim, name)

    def session(self, pm, **kw):
        cfg = self.X.XpConfig.gemma3_1b(n_layers=2, vocab=1024, max_seq=1024, prefill_mode=pm, **kw)
        s = self.X.DecodeSession(cfg)
        s.synthesize(4)
        return s

    def prompt(self, sess, n):
        sess.reset()
        sess.prefill(np.random.default_rng(n).integers(0, 1024, n).astype(np.uint32))
        out = [sess.last_logits().astype(np.float64)]
        out += [sess.kv_download(l, w, 0, n).view(np.float16).astype(np.float64) for l in range(2) for w in (0, 1)]
        return out

    def check(self, sess, n, want):
        for a, b in zip(self.prompt(sess, n), want):
            assert np.abs(a - b).max() <= 1e-3 * np.abs(b).max()

    def limits(self):
        X, limit, allow, largest = self.X, self.var("alloc_limit"), self.var("alloc_allow"), self.var("alloc_largest")
        refused = self.var("alloc_refused", C.c_uint)
        tok = self.session(X.XP_PREFILL_TOKENS)
        want = {n: self.prompt(tok, n) for n in (10, 17, 300)}
        tok.close()
        sizes = {}
        for n in (300, 10):                               # the engine's memory, then the step's
            s = self.session(X.XP_PREFILL_AUTO)
            largest.value = 0
            self.check(s, n, want[n])
            sizes[n] = largest.value
            s.close()
        engine, step = sizes[300], sizes[10]
        print(f"memory: engine {engine} step {step}", flush=True)
        for what, lim, let in (("fewer positions a pass", engine // 2, 0), ("the step only", 0, step), ("token steps only", 0, 0)):
            print(what, flush=True)
            s = self.session(X.XP_PREFILL_AUTO)
            limit.value, allow.value = lim, let
            refused.value, largest.value = 0, 0
            for n in (300, 17, 10, 300):
                self.check(s, n, want[n])
            s.decode_steps(2)
            limit.value = 2 ** 64 - 1
            assert refused.value > 0
            assert {"fewer positions a pass": 4096 < largest.value <= lim}.get(what, largest.value == let), largest.value
            self.check(s, 300, want[300])
            s.close()

    def once(self):
        X, calls = self.X, self.var("alloc_calls", C.c_uint)
        s = self.session(X.XP_PREFILL_AUTO)
        self.prompt(s, 18)
        made = calls.value
        for pos0, n in ((0, 64), (0, 65), (0, 100), (0, 600), (500, 400), (0, 1000), (900, 30)):
            s.set_position(pos0)
            s.prefill(np.arange(n, dtype=np.uint32))
        assert calls.value == made, (calls.value, made)
        s.close()


@pytest.mark.parametrize("hidden,ffn,heads,kvh", [(1152, 6912, 4, 1), (384, 640, 2, 2), (2048, 8192, 4, 2), (8192, 28672, 16, 8)])
def test_prefill_buffers_hold_every_pass(hidden, ffn, heads, kvh):
    """The one allocation against each row count's plans and key splits."""
    lib, total = C.CDLL(os.path.join(ROOT, "tests", "native", "prefill_layout.so")), C.c_uint64()
    for max_seq, rows in ((8192, 2048), (8192, 128), (300, 300), (40, 40)):
        for n_cu in (256, 64):
            assert lib.prefill_layout_misfit(hidden, ffn, heads, kvh, max_seq, rows, n_cu, C.byref(total)) == 0
        assert rows < 2048 or total.value < rows * 20 * (hidden + ffn + 256 * (heads + 2 * kvh))


@pytest.mark.parametrize("rows", [1, 15, 17, 40, 264])
def test_prefill_staging_takes_whole_tiles(rows):
    """Rows that are not whole operand tiles would be updated in place twice."""
    lib = C.CDLL(os.path.join(ROOT, "tests", "native", "prefill_layout.so"))
    assert lib.prefill_staging_rows(rows) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["limits", "once"])
def test_gpu_prefill_low_memory(case):
    print(f"case prefill low memory {case}", flush=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), case], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    getattr(Child(), sys.argv[1])()
    print("ok", flush=True)
