"""The sampling chain's wave-wide selection, tiled exponentials and tiled serial
sums, bit for bit against the oracle where their shapes have edges: chains
shorter and longer than a 1024-element round, ties across the cut and across
rounds, no candidate at all, -inf and NaN elements, more chains than elements,
chain counts around the 16-chain workgroup and the 4096-sum tile, targets in
the first and past the last chain."""
import numpy as np
import pytest

INF, NONE = np.float32(np.inf), 0xFFFFFFFF


def dbuf(X, a):
    return X.DeviceBuffer.from_array(np.ascontiguousarray(a))


def values(kind, n, seed):
    r = np.random.default_rng(seed)
    x = r.normal(0.0, 3.0, n).astype(np.float32)
    if kind == "equal":
        x[:] = 1.5
    elif kind == "few":                       # a handful of distinct values, signed zeros among them
        x = r.choice(np.float32([2.0, 0.0, -0.0, -1.0, 2.0]), n)
    elif kind == "holes":                     # mostly nothing to choose
        x[r.random(n) < 0.97] = -INF
        x[r.random(n) < 0.01] = np.nan
        x[r.integers(0, n, 3)] = INF
    elif kind == "none":
        x[:] = -INF
    elif kind == "rising":
        x = np.arange(n, dtype=np.float32) - np.float32(n // 2)
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "equal", "few", "holes", "none", "rising"])
@pytest.mark.parametrize("n,nparts,k", [(262144, 256, 64), (5000, 1, 64), (70000, 33, 40), (3000, 3, 1),
                                        (1024, 1, 64), (1025, 1, 63), (700, 300, 20), (90, 200, 5),
                                        (60000, 5000, 8)])
def test_gpu_topk_wave_bit_exact(xp, xo, kind, n, nparts, k):
    X, L = xp, xo.lib()
    print(f"case topk wave {kind} n={n} nparts={nparts} k={k}", flush=True)
    x = values(kind, n, n + k)
    nc = nparts * k
    cv, ci = np.empty(nc, np.float32), np.empty(nc, np.uint32)
    L.xo_topk_partial(cv, ci, x, n, nparts, k)
    dv, di, dx = X.DeviceBuffer(4 * nc), X.DeviceBuffer(4 * nc), dbuf(X, x)
    X.call("xp_topk_partial", dv.vp, di.vp, dx.vp, n, nparts, k, None)
    X.synchronize()
    assert np.array_equal(di.download(np.uint32), ci)
    assert np.array_equal(dv.download(np.float32).view(np.uint32), cv.view(np.uint32))
    ov, oi = np.full(k, -7.0, np.float32), np.full(k, 7, np.uint32)
    L.xo_topk_rank_select(ov, oi, cv, ci, nc, k)
    do, dj = dbuf(X, np.full(k, -7.0, np.float32)), dbuf(X, np.full(k, 7, np.uint32))
    X.call("xp_topk_rank_select", do.vp, dj.vp, dv.vp, di.vp, nc, k, None)
    X.synchronize()
    assert np.array_equal(dj.download(np.uint32), oi)
    assert np.array_equal(do.download(np.float32), ov)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "few", "holes"])
@pytest.mark.parametrize("n,nparts,k", [(4096, 256, 1), (24 * 256, 256, 1), (8 * 4096, 4096, 4), (8 * 4096, 4096, 8), (64 * 16384, 16384, 1),
                                        (64 * 4096, 4096, 1), (16 * 16384 - 3, 16384, 8), (16 * 16384, 16384, 16),
                                        (81921 * 16, 81921, 16), (81921 * 16, 81921, 40)])
def test_gpu_topk_partial_both_sides(xp, xo, kind, n, nparts, k):
    """Where the kernels change over: a thread a chain on the first of each
    pair of shapes, a wave a chain on the second."""
    X, L = xp, xo.lib()
    print(f"case topk both sides {kind} n={n} nparts={nparts} k={k}", flush=True)
    x = values(kind, n, n + k)
    nc = nparts * k
    cv, ci = np.empty(nc, np.float32), np.empty(nc, np.uint32)
    L.xo_topk_partial(cv, ci, x, n, nparts, k)
    dv, di, dx = X.DeviceBuffer(4 * nc), X.DeviceBuffer(4 * nc), dbuf(X, x)
    X.call("xp_topk_partial", dv.vp, di.vp, dx.vp, n, nparts, k, None)
    X.synchronize()
    assert np.array_equal(di.download(np.uint32), ci)
    assert np.array_equal(dv.download(np.float32).view(np.uint32), cv.view(np.uint32))


@pytest.mark.gpu
def test_gpu_topk_partial_2_26_chains(xp):
    """A wave for each of 2^26 chains is more than a grid's threads."""
    X = xp
    nparts, rows = 1 << 26, 16
    n = nparts * rows
    print(f"case topk partial nparts={nparts}", flush=True)
    dx, dv, di = X.DeviceBuffer(4 * n), X.DeviceBuffer(4 * nparts), X.DeviceBuffer(4 * nparts)
    dx.fill_bytes(0)
    dv.fill_bytes(0xFF)
    for p, r in ((0, 3), (nparts - 1, 15), (nparts // 2, 0)):
        dx.upload(np.float32([7.0]), 4 * (p + r * nparts))
    X.call("xp_topk_partial", dv.vp, di.vp, dx.vp, n, nparts, 1, None)
    X.synchronize()
    for p, want in ((0, 3 * nparts), (nparts - 1, nparts - 1 + 15 * nparts), (nparts // 2, nparts // 2), (5, 5)):
        assert int(di.download(np.uint32, 1, 4 * p)[0]) == want
        assert float(dv.download(np.float32, 1, 4 * p)[0]) == (0.0 if p == 5 else 7.0)


@pytest.mark.gpu
@pytest.mark.parametrize("nc,k", [(1, 1), (64, 64), (128, 20), (129, 20), (129, 64), (1023, 64), (1025, 3), (16384, 64), (17409, 64), (40000, 64),
                                  (3000, 65), (300, 200)])
def test_gpu_rank_select_any_list(xp, xo, nc, k):
    """Lists in no order: shuffled ids, empty slots, filled -inf slots, the same
    pair twice, ties whose lower id comes later; k above 64 too."""
    X, L = xp, xo.lib()
    print(f"case rank select ncand={nc} k={k}", flush=True)
    r = np.random.default_rng(nc + k)
    cv = r.choice(np.float32(np.linspace(-2, 2, 40)), nc)
    ci = r.permutation(4 * nc)[:nc].astype(np.uint32)
    ci[r.random(nc) < 0.2] = NONE
    cv[r.random(nc) < 0.1] = -INF
    if nc > 10:
        cv[5], ci[5], cv[nc - 2], ci[nc - 2] = 2.5, 77, 2.5, 77
    ov, oi = np.full(k, -7.0, np.float32), np.full(k, 7, np.uint32)
    L.xo_topk_rank_select(ov, oi, cv, ci, nc, k)
    do, dj = dbuf(X, np.full(k, -7.0, np.float32)), dbuf(X, np.full(k, 7, np.uint32))
    dv, di = dbuf(X, cv), dbuf(X, ci)
    X.call("xp_topk_rank_select", do.vp, dj.vp, dv.vp, di.vp, nc, k, None)
    X.synchronize()
    assert np.array_equal(dj.download(np.uint32), oi)
    assert np.array_equal(do.download(np.float32), ov)


@pytest.mark.gpu
@pytest.mark.parametrize("n,nparts", [(5000, 1), (5000, 15), (5000, 17), (100, 100), (4097, 4096), (9000, 4097),
                                      (20000, 8200), (50, 64), (262144, 1024)])
def test_gpu_softmax_and_draw_tiles(xp, xo, n, nparts):
    X, L = xp, xo.lib()
    print(f"case softmax tiles n={n} nparts={nparts}", flush=True)
    x = values("normal", n, nparts)
    dx, dm, ds = dbuf(X, x), X.DeviceBuffer(4 * nparts), dbuf(X, np.zeros(2, np.float32))
    X.call("xp_reduce_max_partial", dm.vp, dx.vp, n, nparts, None)
    X.call("xp_reduce_max_final", ds.vp, dm.vp, nparts, None)
    pm = np.empty(nparts, np.float32)
    L.xo_reduce_max_partial(pm, x, n, nparts)
    dp = X.DeviceBuffer(4 * nparts)
    X.call("xp_softmax_exp_partial", dx.vp, dp.vp, dx.vp, ds.vp, n, nparts, None)   # in place
    X.call("xp_reduce_sum_final", ds.vp, dp.vp, nparts, None)
    X.synchronize()
    assert np.array_equal(dm.download(np.float32), pm)
    st, e, ps = ds.download(np.float32), dx.download(np.float32), dp.download(np.float32)
    assert st[0] == x.max()
    # the device's exponentials summed in chain order, then in chain-sum order
    assert np.allclose(e, np.exp(x.astype(np.float64) - float(st[0])), rtol=2e-6, atol=1e-30)
    want = np.empty(nparts, np.float32)
    L.xo_reduce_sum_partial(want, e, n, nparts)
    assert np.array_equal(ps, want)
    s2 = np.zeros(2, np.float32)
    L.xo_reduce_sum_final(s2, ps, nparts)
    assert st[1] == s2[1]
    if nparts > n:
        return
    do, di = X.DeviceBuffer(8), X.DeviceBuffer(4)
    for u in (0.0, 1e-7, 0.31, 0.5, 0.93, 0.999999, 1.0, 1.5, -0.5):
        X.call("xp_multinomial_strided", do.vp, di.vp, dx.vp, dp.vp, ds.vp, n, nparts, u, None)
        X.synchronize()
        out, oi = np.empty(2, np.float32), np.empty(1, np.uint32)
        L.xo_multinomial_strided(out, oi, e, ps, st, n, nparts, np.float32(u))
        assert int(di.download(np.uint32)[0]) == int(oi[0]), u
        assert np.array_equal(do.download(np.float32), out), u


@pytest.mark.gpu
@pytest.mark.parametrize("n,nparts", [(1, 1), (15, 1), (16, 1), (17, 1), (63, 1), (64, 1), (65, 1), (80, 1), (1000, 1), (129, 2), (1000, 31)])
def test_gpu_draw_inside_a_chain(xp, xo, n, nparts):
    """The walk inside the chosen chain (64 elements at a time, the last few of
    a chain one by one): targets on, before and past every element's running sum."""
    X, L = xp, xo.lib()
    print(f"case draw inside a chain n={n} nparts={nparts}", flush=True)
    w = np.random.default_rng(n).random(n).astype(np.float32)
    w[::5] = 0.0
    ps = np.empty(nparts, np.float32)
    L.xo_reduce_sum_partial(ps, w, n, nparts)
    st = np.float32([0.0, 1.0])                          # u is the target itself
    dw, dp, ds, do, di = dbuf(X, w), dbuf(X, ps), dbuf(X, st), X.DeviceBuffer(8), X.DeviceBuffer(4)
    run = np.cumsum(w[::nparts], dtype=np.float32)
    us = np.unique(np.concatenate([run[:3], run[14:18], run[62:66], run[-2:], np.float32([0.0, -1.0, 1e6])]))
    for u in np.concatenate([us, np.nextafter(us, np.float32(1e9))]):
        out, oi = np.empty(2, np.float32), np.empty(1, np.uint32)
        L.xo_multinomial_strided(out, oi, w, ps, st, n, nparts, u)
        X.call("xp_multinomial_strided", do.vp, di.vp, dw.vp, dp.vp, ds.vp, n, nparts, float(u), None)
        X.synchronize()
        assert int(di.download(np.uint32)[0]) == int(oi[0]), u
        assert np.array_equal(do.download(np.float32), out), u


@pytest.mark.gpu
@pytest.mark.parametrize("n,nparts", [(16 * 300 - 1, 300), (16 * 300, 300), (24 * 300 - 1, 300), (24 * 300, 300), (131071 * 24, 131071),
                                      (131072 * 25 + 5, 131072), (65536 * 17, 65536), (65536 * 16 + 1, 65536), (7, 1000)])
def test_gpu_chain_partials_both_sides(xp, xo, n, nparts):
    """Maxima and exponential sums where the kernels change over (a thread a
    chain, sixteen a chain): bit for bit the oracle's of the device's exponentials."""
    X, L = xp, xo.lib()
    print(f"case chain partials n={n} nparts={nparts}", flush=True)
    x = values("normal", n, nparts)
    x[::97] = -INF
    dx, dm, ds = dbuf(X, x), X.DeviceBuffer(4 * nparts), dbuf(X, np.float32([x.max(), 0.0]))
    do, dp = X.DeviceBuffer(4 * n), X.DeviceBuffer(4 * nparts)
    X.call("xp_reduce_max_partial", dm.vp, dx.vp, n, nparts, None)
    X.call("xp_softmax_exp_partial", do.vp, dp.vp, dx.vp, ds.vp, n, nparts, None)
    X.synchronize()
    pm, want = np.empty(nparts, np.float32), np.empty(nparts, np.float32)
    L.xo_reduce_max_partial(pm, x, n, nparts)
    assert np.array_equal(dm.download(np.float32), pm)
    e = do.download(np.float32)
    assert np.allclose(e, np.exp(x.astype(np.float64) - float(x.max())), rtol=2e-6, atol=1e-30)
    L.xo_reduce_sum_partial(want, e, n, nparts)
    assert np.array_equal(dp.download(np.float32), want)


@pytest.mark.gpu
def test_gpu_chain_partials_past_2_28_chains(xp):
    """Sixteen threads for each of 2^28 chains are more than a grid has."""
    X = xp
    nparts = (1 << 28) + 64
    n = nparts + 3
    print(f"case chain partials nparts={nparts}", flush=True)
    dx, dm, ds = X.DeviceBuffer(4 * n), X.DeviceBuffer(4 * nparts), dbuf(X, np.float32([0.0, 0.0]))
    dx.fill_bytes(0)
    dm.fill_bytes(0xFF)
    dx.upload(np.float32([5.0]), 4 * (nparts - 1))
    X.call("xp_reduce_max_partial", dm.vp, dx.vp, n, nparts, None)
    X.synchronize()
    for off, want in ((0, [0.0] * 5), (4 * (nparts - 3), [0.0, 0.0, 5.0])):
        assert np.array_equal(dm.download(np.float32, len(want), off), np.float32(want))
    X.call("xp_softmax_exp_partial", dx.vp, dm.vp, dx.vp, ds.vp, n, nparts, None)
    X.synchronize()
    assert np.array_equal(dm.download(np.float32, 5), np.float32([2, 2, 2, 1, 1]))
    assert np.array_equal(dm.download(np.float32, 2, 4 * (nparts - 3)), np.float32([1, 1]))
    assert np.array_equal(dx.download(np.float32, 3, 4 * nparts), np.float32([1, 1, 1]))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 63, 64, 65, 200])
def test_gpu_topp_and_draw_any_k(xp, xo, k):
    X, L = xp, xo.lib()
    print(f"case topp / draw k={k}", flush=True)
    r = np.random.default_rng(k)
    w0 = np.sort(r.random(k).astype(np.float32))[::-1].copy()
    ids = r.permutation(100000)[:k].astype(np.uint32)
    dids = dbuf(X, ids)
    for p in (0.05, 0.7, 1.0):
        w = w0.copy()
        L.xo_topp_cutoff(w, k, np.float32(p))
        dw = dbuf(X, w0)
        X.call("xp_topp_cutoff", dw.vp, k, p, None)
        X.synchronize()
        assert np.array_equal(dw.download(np.float32), w)
        do, di = X.DeviceBuffer(8), X.DeviceBuffer(4)
        for u in (0.0, 0.2, 0.77, 1.0, 2.0):
            out, oi = np.empty(2, np.float32), np.empty(1, np.uint32)
            L.xo_multinomial_sample(out, oi, w, ids, k, np.float32(u))
            X.call("xp_multinomial_sample", do.vp, di.vp, dw.vp, dids.vp, k, u, None)
            X.synchronize()
            assert int(di.download(np.uint32)[0]) == int(oi[0]) and np.array_equal(do.download(np.float32), out)


def terms(kind, n, seed):
    r = np.random.default_rng(seed)
    if kind == "even":                        # a softmax's chain sums
        return r.uniform(0.5, 1.5, n).astype(np.float32)
    if kind == "wide":
        return np.exp(r.normal(0, 6, n)).astype(np.float32)
    if kind == "ties":                        # whole numbers and halves of the sum's last place, on both sides of even
        return np.concatenate([np.float32([2.0 ** 23 + 1]), r.integers(0, 6, n).astype(np.float32) / 2])[:n]
    if kind == "tiny":                        # denormal terms and sums
        return (r.integers(0, 1 << 22, n).astype(np.uint32)).view(np.float32)
    x = np.where(r.random(n) < 0.8, 0.0, r.random(n)).astype(np.float32)
    if kind == "signs":
        x -= np.float32(0.05)
        x[::7] = -0.0
    elif kind == "inf":
        x[n // 2] = np.inf
    elif kind == "nan":
        x[2 * n // 3] = np.nan
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["even", "wide", "ties", "tiny", "sparse", "signs", "inf", "nan"])
@pytest.mark.parametrize("n", [1, 63, 64, 257, 4096, 4100, 9000])
def test_gpu_serial_sums_bit_exact(xp, xo, kind, n):
    """The sums and the place in them, which are formed in blocks, against the
    oracle's one chain of adds."""
    X, L = xp, xo.lib()
    print(f"case serial sums {kind} n={n}", flush=True)
    w = terms(kind, n, n)
    dw, ds = dbuf(X, w), dbuf(X, np.zeros(2, np.float32))
    X.call("xp_reduce_sum_final", ds.vp, dw.vp, n, None)
    X.synchronize()
    want = np.zeros(2, np.float32)
    L.xo_reduce_sum_final(want, w, n)
    assert np.array_equal(ds.download(np.float32), want, equal_nan=True)
    do, di = X.DeviceBuffer(8), X.DeviceBuffer(4)
    for u in (0.0, 0.013, 0.24, 0.5000001, 0.77, 0.9999, 1.0, 1.01, -1.0):
        X.call("xp_multinomial_strided", do.vp, di.vp, dw.vp, dw.vp, ds.vp, n, n, u, None)
        X.synchronize()
        out, oi = np.empty(2, np.float32), np.empty(1, np.uint32)
        L.xo_multinomial_strided(out, oi, w, w, want, n, n, np.float32(u))
        assert int(di.download(np.uint32)[0]) == int(oi[0]), u
        assert np.array_equal(do.download(np.float32), out, equal_nan=True), u
