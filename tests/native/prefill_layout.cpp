// The prompt prefill's one allocation against what its passes need, on the host.
// Names of its own: the library's must not resolve to this copy.
#define PrefillEngine LayoutTestEngine
#define prefill_engine_create layout_test_engine_create
#define prefill_engine_run layout_test_engine_run
#define prefill_engine_destroy layout_test_engine_destroy
#include "../../xpose_amd/csrc/prefill.cpp"

// The first row count up to the layout's whose pass does not fit its buffers,
// alone or at any depth of the context; 0: all fit.
extern "C" uint32_t prefill_layout_misfit(uint32_t hidden, uint32_t ffn, uint32_t n_heads, uint32_t n_kv_heads,
                                          uint32_t max_seq, uint32_t rows, int n_cu, uint64_t* total) {
    xp_config c{};
    c.hidden = hidden;
    c.ffn = ffn;
    c.n_heads = n_heads;
    c.n_kv_heads = n_kv_heads;
    c.head_dim = 256;
    c.max_seq = max_seq;
    const xp::PfLayout l = xp::plan_layout(c, n_cu, rows);
    const size_t offs[] = {l.ids, l.x, l.a, l.asum, l.a2, l.asum2, l.qkv, l.y, l.qh, l.ql, l.qscale, l.part, l.total};
    for (int i = 0; i < 12; ++i)
        if (offs[i] > offs[i + 1]) return ~0u;
    *total = l.total;
    const uint32_t G = n_heads / n_kv_heads, qd = n_heads * 256u;
    for (uint32_t r = 1; r <= rows; ++r) {
        const xp::PfPass p = xp::plan_pass(c, n_cu, r);
        bool ok = p.qkv_floats <= l.qkv_floats && p.y_floats <= l.y_floats && size_t(p.pad) * hidden * 4 <= l.a - l.x &&
                  size_t(p.pad) * std::max(hidden, qd) * 4 <= l.asum - l.a && size_t(p.pad) * std::max(hidden, qd) / 8 <= l.a2 - l.asum &&
                  size_t(p.pad) * ffn * 4 <= l.asum2 - l.a2 && size_t(p.pad) * ffn / 8 <= l.qkv - l.asum2 &&
                  l.qkv_floats * 4 <= l.y - l.qkv && l.y_floats * 4 <= l.qh - l.y && l.part_floats * 4 <= l.total - l.part;
        for (uint32_t keys = r; keys <= max_seq; keys += 64u) {
            const uint32_t z = xp::pf_attn_splits(r, G, n_kv_heads, keys, n_cu);
            ok = ok && (z == 1u || size_t(n_kv_heads) * ((r * G + 31u) / 32u) * z * 32u * xp::kPfRecord <= l.part_floats);
        }
        if (!ok) return r;
    }
    return 0;
}

// launch_pf_prep's answer to a row count (nothing is launched for one it refuses).
extern "C" int prefill_staging_rows(uint32_t rows_pad) {
    xp::PfPrepArgs a{};
    a.K = 1152;
    a.rows_pad = rows_pad;
    return xp::launch_pf_prep(a, nullptr);
}
