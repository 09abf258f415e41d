// Prompt prefill of a decode session: the stages of prefill_engine.hip over
// chunks of up to kPfMaxRows positions. The reference prefills one token step
// at a time (DecodeSession::prefill, examples/llm/decode.cpp:1785-1815); the
// KV rows and logits are the same to rounding.
//
// Plain launches on the session's stream: a stage takes about as long as its
// launch or longer, so the host stays ahead. The buffers are one allocation,
// made at the first prompt for the most positions a pass can have (kPfMaxRows
// or the session's context: 177 MB for 2048 at hidden 1152 and ffn 6912; half
// as many while the device refuses it). No prompt allocates, frees or waits
// after that. A first prompt of 32 tokens pays about 0.05 ms for it.
#include "xp_internal.hpp"
#include "xp_launch.hpp"

#include <algorithm>
#include <new>

namespace xp {

namespace {
constexpr size_t kAlignP = 256;
constexpr uint32_t kBlkP = 32;   // quantisation block along k
size_t al(size_t v) { return (v + kAlignP - 1) & ~(kAlignP - 1); }
}  // namespace

// The buffers of a pass: byte offsets in the arena, and the floats that the
// three of them take whose size depends on a plan's splits.
struct PfLayout {
    uint32_t rows = 0;           // most positions of a pass
    size_t ids, x, a, asum, a2, asum2, qkv, y, qh, ql, qscale, part, total;
    size_t qkv_floats = 0, y_floats = 0, part_floats = 0;
};

struct PrefillEngine {
    const xp_session* owner = nullptr;
    SessionWeights w{};
    hipStream_t st = nullptr;    // the owner's stream, during a run
    char* arena = nullptr;
    PfLayout lay;

    int chunk(const uint32_t* ids_dev, uint32_t rows, uint32_t pos0);
};

namespace {

// What a pass of `rows` positions runs: its GEMMs' plans and padded rows.
struct PfPass {
    PfGemmPlan q, o, g, d;
    bool wide;                   // operand tiles of 32 rows, for the 128-row GEMM, else of 16
    uint32_t pad;                // rows in whole operand tiles
    size_t qkv_floats, y_floats;
};
PfPass plan_pass(const xp_config& c, int n_cu, uint32_t rows) {
    const uint32_t H = c.hidden, F = c.ffn, qd = c.n_heads * c.head_dim, N = qd + 2 * c.n_kv_heads * c.head_dim;
    PfPass p;
    p.q = plan_pf_gemm(rows, N, H / kBlkP, false, n_cu);
    p.o = plan_pf_gemm(rows, H, qd / kBlkP, false, n_cu);
    p.g = plan_pf_gemm(rows, F, H / kBlkP, true, n_cu);
    p.d = plan_pf_gemm(rows, H, F / kBlkP, false, n_cu);
    p.wide = p.q.shape == 2;
    p.pad = p.wide ? (rows + 31u) / 32u * 32u : (rows + 15u) / 16u * 16u;
    p.qkv_floats = size_t(p.pad) * N * p.q.splits;
    p.y_floats = size_t(p.pad) * H * std::max(p.o.splits, p.d.splits);
    return p;
}

PfLayout plan_layout(const xp_config& c, int n_cu, uint32_t rows) {
    const uint32_t H = c.hidden, F = c.ffn, qd = c.n_heads * c.head_dim;
    PfLayout l;
    l.rows = rows;
    // The row counts up to hi that have as many row tiles as hi: their plans
    // split no more than the fewest rows' (partial sums cost by the row), and
    // hi pads to the most.
    for (uint32_t lo = 1, hi; lo <= rows; lo = hi + 1u) {
        hi = std::min(lo <= 32u ? 32u : lo <= 64u ? 64u : (lo + 127u) / 128u * 128u, rows);
        const PfPass a = plan_pass(c, n_cu, lo), b = plan_pass(c, n_cu, hi);
        const size_t pad = std::max(a.pad, b.pad);
        l.qkv_floats = std::max({l.qkv_floats, a.qkv_floats / a.pad * pad, b.qkv_floats});
        l.y_floats = std::max({l.y_floats, a.y_floats / a.pad * pad, b.y_floats});
    }
    // key splits only add workgroups up to one a CU
    if (pf_attn_splits(1, 1, 1, c.max_seq, n_cu) > 1u) l.part_floats = size_t(std::max(n_cu, 256)) * 32u * kPfRecord;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += al(bytes); return o; };
    const size_t pad = (rows + 31u) / 32u * 32u;
    l.ids = take(size_t(c.max_seq) * 4);
    l.x = take(pad * H * 4);
    l.a = take(pad * std::max(H, qd) * 4);
    l.asum = take(pad * std::max(H, qd) / 8);
    l.a2 = take(pad * F * 4);
    l.asum2 = take(pad * F / 8);
    l.qkv = take(l.qkv_floats * 4);
    l.y = take(l.y_floats * 4);
    l.qh = take(size_t(rows) * qd * 2);
    l.ql = take(size_t(rows) * qd * 2);
    l.qscale = take(size_t(rows) * c.n_heads * 4);
    l.part = take(l.part_floats * 4);
    l.total = off;
    return l;
}

}  // namespace

int PrefillEngine::chunk(const uint32_t* ids_dev, uint32_t rows, uint32_t pos0) {
    const xp_config& c = w.cfg;
    const uint32_t H = c.hidden, F = c.ffn, qd = c.n_heads * c.head_dim, kvd = c.n_kv_heads * c.head_dim;
    const uint32_t G = c.n_heads / c.n_kv_heads, N = qd + 2 * kvd;
    const PfPass ps = plan_pass(c, w.n_cu, rows);
    const PfGemmPlan &pq = ps.q, &po = ps.o, &pg = ps.g, &pd = ps.d;
    const bool wide = ps.wide;
    const uint32_t pad = ps.pad, mt = pad / 16u;
    const uint32_t zs_g = pf_attn_splits(rows, G, c.n_kv_heads, pos0 + rows, w.n_cu);
    const uint32_t loc_keys = c.sliding_window ? std::min(pos0 + rows, c.sliding_window + 32u) : pos0 + rows;
    const uint32_t zs_l = pf_attn_splits(rows, G, c.n_kv_heads, loc_keys, w.n_cu), zs = std::max(zs_g, zs_l);
    const size_t part = zs > 1u ? size_t(c.n_kv_heads) * ((rows * G + 31u) / 32u) * zs * 32u * kPfRecord : 0;
    if (rows > lay.rows || ps.qkv_floats > lay.qkv_floats || ps.y_floats > lay.y_floats || part > lay.part_floats)
        return set_error(XP_E_NOMEM, "prefill: %u positions do not fit the buffers", rows);
    const size_t o_x = lay.x, o_a = lay.a, o_as = lay.asum, o_a2 = lay.a2, o_as2 = lay.asum2, o_qkv = lay.qkv, o_y = lay.y,
                 o_qh = lay.qh, o_ql = lay.ql, o_qs = lay.qscale, o_part = lay.part;
    auto f = [&](size_t o) { return reinterpret_cast<float*>(arena + o); };
    float* x = f(o_x);
    int rc;
#define XB(call) do { if ((rc = (call)) != XP_OK) return rc; } while (0)
    PfPrepArgs pr{};
    pr.x = x;
    pr.w_pre = w.layer[0].norm[0];
    pr.a = arena + o_a;
    pr.asum = f(o_as);
    pr.K = H;
    pr.rows = rows;
    pr.rows_pad = pad;
    pr.wide = wide;
    pr.eps = c.rms_eps;
    pr.tok = ids_dev;
    pr.ewq = w.lm_w;
    pr.esc = w.lm_s;
    pr.etable = w.embed;
    pr.vocab = c.vocab;
    pr.efmt = c.scale_fmt;
    pr.escale = w.embed_scale;
    XB(launch_pf_prep(pr, st));
    pr.tok = nullptr;
    PfGemmArgs base{};
    base.a = arena + o_a;
    base.asum = f(o_as);
    base.m_tiles = mt;
    for (uint32_t l = 0; l < c.n_layers; ++l) {
        const SessionWeights::Layer& L = w.layer[l];
        PfGemmArgs g = base;
        g.mats[0] = {nullptr, L.w[XP_T_Q], L.s[XP_T_Q], qd};
        g.mats[1] = {nullptr, L.w[XP_T_K], L.s[XP_T_K], kvd};
        g.mats[2] = {nullptr, L.w[XP_T_V], L.s[XP_T_V], kvd};
        g.n_mats = 3;
        g.nblk = H / kBlkP;
        g.out = f(o_qkv);
        g.ldo = N;
        XB(launch_pf_gemm(g, pq, c.scale_fmt, false, st, "prefill qkv"));
        PfQkArgs qa{};
        qa.qkv = f(o_qkv);
        qa.splits = pq.splits;
        qa.rows = rows;
        qa.rows_pad = pad;
        qa.n_heads = c.n_heads;
        qa.kv_heads = c.n_kv_heads;
        qa.pos0 = pos0;
        qa.qw = L.norm[4];
        qa.kw = L.norm[5];
        qa.eps = c.rms_eps;
        qa.kc = L.kc;
        qa.vc = L.vc;
        qa.qh = reinterpret_cast<_Float16*>(arena + o_qh);
        qa.ql = reinterpret_cast<_Float16*>(arena + o_ql);
        qa.qscale = f(o_qs);
        XB(launch_pf_qk(qa, L.global ? c.rope_theta_global : c.rope_theta_local, st));
        // the last layer's KV rows are the last thing a prefill produces
        if (l + 1 == c.n_layers) break;
        PfAttnArgs aa{};
        aa.qh = qa.qh;
        aa.ql = qa.ql;
        aa.qscale = qa.qscale;
        aa.kc = L.kc;
        aa.vc = L.vc;
        aa.rows = rows;
        aa.kv_heads = c.n_kv_heads;
        aa.pos0 = pos0;
        aa.window = L.global ? 0u : c.sliding_window;
        aa.scale = w.attn_scale;
        aa.a = arena + o_a;
        aa.asum = f(o_as);
        aa.nblk = qd / kBlkP;
        aa.wide = wide;
        aa.part = f(o_part);
        XB(launch_pf_attn(aa, G, L.global ? zs_g : zs_l, st));
        g = base;
        g.mats[0] = {nullptr, L.w[XP_T_O], L.s[XP_T_O], H};
        g.n_mats = 1;
        g.nblk = qd / kBlkP;
        g.out = f(o_y);
        g.ldo = H;
        XB(launch_pf_gemm(g, po, c.scale_fmt, false, st, "prefill o_proj"));
        pr.y = f(o_y);
        pr.ysplit = po.splits;
        pr.w_post = L.norm[1];
        pr.w_pre = L.norm[2];
        XB(launch_pf_prep(pr, st));
        g = base;
        g.mats[0] = {nullptr, L.w[XP_T_GATE], L.s[XP_T_GATE], F};
        g.mats[1] = {nullptr, L.w[XP_T_UP], L.s[XP_T_UP], F};
        g.n_mats = 2;
        g.nblk = H / kBlkP;
        g.a_out = arena + o_a2;
        g.asum_out = f(o_as2);
        g.nblk_out = F / kBlkP;
        XB(launch_pf_gemm(g, pg, c.scale_fmt, true, st, "prefill gate/up"));
        g = base;
        g.a = arena + o_a2;
        g.asum = f(o_as2);
        g.mats[0] = {nullptr, L.w[XP_T_DOWN], L.s[XP_T_DOWN], H};
        g.n_mats = 1;
        g.nblk = F / kBlkP;
        g.out = f(o_y);
        g.ldo = H;
        XB(launch_pf_gemm(g, pd, c.scale_fmt, false, st, "prefill down"));
        pr.ysplit = pd.splits;
        pr.w_post = L.norm[3];
        pr.w_pre = w.layer[l + 1].norm[0];
        XB(launch_pf_prep(pr, st));
    }
#undef XB
    return XP_OK;
}

int prefill_engine_create(const xp_session* s, PrefillEngine** out) {
    *out = nullptr;
    PrefillEngine* p = new (std::nothrow) PrefillEngine;
    if (!p) return set_error(XP_E_NOMEM, "prefill: out of host memory");
    p->owner = s;
    if (int rc = session_weights(s, &p->w); rc != XP_OK) {
        delete p;
        return rc;
    }
    const xp_config& c = p->w.cfg;
    const uint32_t G = c.n_kv_heads && c.n_heads % c.n_kv_heads == 0 ? c.n_heads / c.n_kv_heads : 0;
    const char* why = nullptr;
    if (c.scale_fmt != XP_SCALE_F16_QUAD && c.scale_fmt != XP_SCALE_BF16_QUAD) why = "takes fp16 or bf16 quad scales";
    else if (c.head_dim != 256u || (G != 1u && G != 2u && G != 4u)) why = "takes 1, 2 or 4 query heads of 256 dims per kv head";
    else if (c.hidden % 128u || c.ffn % 128u || c.hidden > 8192u) why = "takes hidden and ffn sizes that are multiples of 128";
    else if (size_t(c.hidden) * c.ffn / 2 > 0xFFFFFFFFu || c.ffn > 1u << 24) why = "takes matrices of up to 4 GiB";
    if (why) {
        delete p;
        return set_error(XP_E_ARG, "prefill: the batched path %s", why);
    }
    // the GEMMs' byte offsets into a staged operand are 32 bits
    const size_t k = std::max({c.hidden, c.ffn, c.n_heads * c.head_dim});
    const uint32_t most = uint32_t(std::min<size_t>(std::min(kPfMaxRows, c.max_seq), 0xFFFFFFFFu / (k * 4u) / 32u * 32u));
    for (uint32_t rows = most;; rows /= 2u) {
        p->lay = plan_layout(c, p->w.n_cu, rows);
        if (hipMalloc(reinterpret_cast<void**>(&p->arena), p->lay.total) == hipSuccess) break;
        p->arena = nullptr;
        const int rc = set_error(XP_E_NOMEM, "prefill: device memory (%zu bytes)", p->lay.total);
        if (rows <= 64u) {
            delete p;
            return rc;
        }
    }
    clear_error();
    *out = p;
    return XP_OK;
}

int prefill_engine_run(PrefillEngine* p, const uint32_t* ids, uint32_t n, uint32_t pos0, hipStream_t st) {
    p->st = st;
    // the weights as they are now: an embedding table may have been uploaded
    // since the last run
    if (int rc = session_weights(p->owner, &p->w); rc != XP_OK) return rc;
    uint32_t* d_ids = reinterpret_cast<uint32_t*>(p->arena + p->lay.ids);
    XP_HIP(hipMemcpyAsync(d_ids, ids, size_t(n) * 4, hipMemcpyHostToDevice, st));
    for (uint32_t c0 = 0; c0 < n;) {
        const uint32_t rows = std::min(p->lay.rows, n - c0);
        if (int rc = p->chunk(d_ids + c0, rows, pos0 + c0); rc != XP_OK) {
            (void)hipStreamSynchronize(st);
            return rc;
        }
        c0 += rows;
    }
    return XP_OK;
}

void prefill_engine_destroy(PrefillEngine* p) {
    if (!p) return;
    if (p->arena) (void)hipFree(p->arena);
    delete p;
}

}  // namespace xp
