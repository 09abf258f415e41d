"""The prefill twins' tiled kernels at the edges of their tiles (32 x 64 scores,
32 rows x 64 or 128 dims of the apply, 256 keys a pass, 2048 held softmax columns),
against the oracle: partly filled tiles, tiles that cross from one head to the
next, several kv heads, head sizes that are no multiple of a chunk, rows that
are not 16-byte aligned, probabilities that are zero where v is not finite.
Tolerance 1e-5 of the largest magnitude (float32 sums in another order), masks
and non-finite places exact, as in tests/test_prefill_kernels.py."""
import numpy as np
import pytest


def dev(X, a):
    return X.DeviceBuffer.from_array(np.ascontiguousarray(a))


def close(got, want):
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    if fin.any():
        assert np.abs(got[fin].astype(np.float64) - want[fin]).max() <= 1e-5 * max(np.abs(want[fin]).max(), 1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh,hd,nq,seq,off,window", [
    (4, 1, 256, 1, 1, 0, 0), (4, 1, 256, 1, 700, 699, 0), (4, 1, 256, 16, 64, 48, 0), (4, 1, 256, 17, 65, 48, 20),
    (4, 1, 256, 200, 200, 0, 0), (4, 1, 256, 129, 640, 511, 100), (4, 2, 128, 33, 97, 64, 0), (6, 2, 36, 50, 130, 80, 7),
    (3, 3, 64, 64, 64, 0, 1), (2, 1, 20, 5, 300, 100, 0), (1, 1, 260, 70, 71, 3, 0),
    (8, 4, 260, 700, 400, 0, 90), (8, 8, 64, 1, 4500, 4499, 0), (8, 8, 64, 3, 4500, 4497, 512), (8, 2, 64, 60, 2100, 2040, 0)])
def test_gpu_prefill_scores_and_apply_tiles(xp, xo, heads, kvh, hd, nq, seq, off, window):
    X, L = xp, xo.lib()
    print(f"case prefill tiles {heads}/{kvh} hd={hd} nq={nq} seq={seq} off={off} window={window}", flush=True)
    r = np.random.default_rng(seq * 7 + nq)
    q, k, v = (r.uniform(-1, 1, n).astype(np.float32) for n in (heads * nq * hd, seq * kvh * hd, seq * kvh * hd))
    want = np.empty(heads * nq * seq, np.float32)
    L.xo_attention_scores_prefill(want, q, k, heads, kvh, hd, nq, seq, off, window, np.float32(0.25))
    ds, dq, dk, dv = dev(X, np.full(want.size, -1e30, np.float32)), dev(X, q), dev(X, k), dev(X, v)
    X.call("xp_attention_scores_prefill", ds.vp, dq.vp, dk.vp, heads, kvh, hd, nq, seq, off, window, 0.25, None)
    X.synchronize()
    close(ds.download(np.float32), want)
    st = np.empty(2 * heads * nq, np.float32)
    L.xo_softmax_rows_stats(st, want, heads * nq, seq)
    L.xo_softmax_rows_apply(want, st, heads * nq, seq)
    dp = dev(X, want)
    out = np.empty(heads * nq * hd, np.float32)
    for case in ("plain", "not finite", "unaligned"):
        if case == "not finite":             # in rows no query, and in rows some queries give any weight
            v = v.copy()
            v[r.integers(0, v.size, 1 + v.size // 4000)] = r.choice(np.float32([np.inf, -np.inf, np.nan]))
            dv = dev(X, v)
        shift = 4 if case == "unaligned" else 0
        L.xo_attention_apply_prefill(out, want, v, heads, kvh, hd, nq, seq)
        do = X.DeviceBuffer(4 * out.size + 16)
        X.call("xp_attention_apply_prefill", do.ptr + shift, dp.vp, dv.vp, heads, kvh, hd, nq, seq, None)
        X.synchronize()
        close(do.download(np.float32, out.size, shift), out)


@pytest.mark.gpu
def test_gpu_prefill_apply_any_head_dim(xp, xo):
    X, L = xp, xo.lib()
    print("case prefill apply head_dim 6", flush=True)
    r = np.random.default_rng(6)
    p, v = r.random(2 * 5 * 40).astype(np.float32), r.uniform(-1, 1, 40 * 6).astype(np.float32)
    out = np.empty(2 * 5 * 6, np.float32)
    L.xo_attention_apply_prefill(out, p, v, 2, 1, 6, 5, 40)
    do, dp, dv = X.DeviceBuffer(4 * out.size), dev(X, p), dev(X, v)
    X.call("xp_attention_apply_prefill", do.vp, dp.vp, dv.vp, 2, 1, 6, 5, 40, None)
    X.synchronize()
    close(do.download(np.float32), out)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 63), (3, 65), (9, 513), (4, 2047), (4, 2048), (6, 2049), (2, 9000),
                                       (7, 64), (7, 128), (7, 129), (7, 257), (7, 1024), (7, 1025), (9000, 191), (9000, 192), (900, 1748)])
def test_gpu_softmax_rows_lengths(xp, rows, cols):
    X = xp
    print(f"case softmax rows {rows} x {cols}", flush=True)
    x = np.random.default_rng(cols).normal(0, 4, rows * cols).astype(np.float32)
    x[1::3] = -np.inf
    if rows > 1:
        x[cols:2 * cols] = -np.inf
    dx, ds = dev(X, x), X.DeviceBuffer(8 * rows)
    X.call("xp_softmax_rows_stats", ds.vp, dx.vp, rows, cols, None)
    X.call("xp_softmax_rows_apply", dx.vp, ds.vp, rows, cols, None)
    X.synchronize()
    # against float64 (the oracle adds a row serially, which at 9000 columns is
    # itself further off than the kernel): a lane adds cols / 64 terms, the wave
    # six times more, each within 2^-24 of the positive sum; the exponential,
    # its argument's subtraction and the division within 4e-6
    tol = (cols / 64 + 8) * 2.0 ** -24 + 4e-6
    x64 = x.reshape(rows, cols).astype(np.float64)
    top = x64.max(1)
    live = np.isfinite(top)
    st, got = ds.download(np.float32).reshape(rows, 2), dx.download(np.float32).reshape(rows, cols)
    assert np.array_equal(st[~live], np.tile(np.float32([0, 1]), ((~live).sum(), 1))) and not got[~live].any()
    e = np.exp(x64[live] - top[live, None])
    assert np.array_equal(st[live, 0], top[live].astype(np.float32))
    assert np.abs(st[live, 1] / e.sum(1) - 1).max() <= tol
    want = e / e.sum(1, keepdims=True)
    assert np.abs(got[live] - want).max() <= 2 * tol * want.max()
