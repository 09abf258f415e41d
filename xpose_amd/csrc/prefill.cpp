// Prompt prefill of a decode session: the stages of prefill_engine.hip over
// chunks of up to kPfMaxRows positions. The reference prefills one token step
// at a time (DecodeSession::prefill, examples/llm/decode.cpp:1785-1815); the
// KV rows and logits are the same to rounding.
//
// Plain launches on the session's stream: a stage takes about as long as its
// launch or longer, so the host stays ahead. The buffers grow with the longest
// chunk seen.
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

struct PrefillEngine {
    const xp_session* owner = nullptr;
    SessionWeights w{};
    hipStream_t st = nullptr;    // the owner's stream, during a run
    char* arena = nullptr;
    size_t arena_bytes = 0;
    uint32_t* d_ids = nullptr;   // [max_seq]

    int chunk(const uint32_t* ids_dev, uint32_t rows, uint32_t pos0);
    int reserve(size_t bytes);
};

int PrefillEngine::reserve(size_t bytes) {
    if (bytes <= arena_bytes) return XP_OK;
    XP_HIP(hipStreamSynchronize(st));
    if (arena) (void)hipFree(arena);
    arena = nullptr;
    arena_bytes = 0;
    if (hipMalloc(reinterpret_cast<void**>(&arena), bytes) != hipSuccess) {
        arena = nullptr;
        return set_error(XP_E_NOMEM, "prefill: device memory (%zu bytes)", bytes);
    }
    arena_bytes = bytes;
    return XP_OK;
}

int PrefillEngine::chunk(const uint32_t* ids_dev, uint32_t rows, uint32_t pos0) {
    const xp_config& c = w.cfg;
    const uint32_t H = c.hidden, F = c.ffn, qd = c.n_heads * c.head_dim, kvd = c.n_kv_heads * c.head_dim;
    const uint32_t G = c.n_heads / c.n_kv_heads, N = qd + 2 * kvd;
    // whole operand tiles: of 32 rows for the 128-row GEMM, else of 16
    const bool wide = plan_pf_gemm(rows, H, H / kBlkP, false, w.n_cu).shape == 2;
    const uint32_t pad = wide ? (rows + 31u) / 32u * 32u : (rows + 15u) / 16u * 16u, mt = pad / 16u;
    const PfGemmPlan pq = plan_pf_gemm(rows, N, H / kBlkP, false, w.n_cu), po = plan_pf_gemm(rows, H, qd / kBlkP, false, w.n_cu),
                     pg = plan_pf_gemm(rows, F, H / kBlkP, true, w.n_cu), pd = plan_pf_gemm(rows, H, F / kBlkP, false, w.n_cu);
    const uint32_t zs_g = pf_attn_splits(rows, G, c.n_kv_heads, pos0 + rows, w.n_cu);
    const uint32_t loc_keys = c.sliding_window ? std::min(pos0 + rows, c.sliding_window + 32u) : pos0 + rows;
    const uint32_t zs_l = pf_attn_splits(rows, G, c.n_kv_heads, loc_keys, w.n_cu);
    // buffers of this chunk
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += al(bytes); return o; };
    const size_t o_x = take(size_t(pad) * H * 4), o_a = take(size_t(pad) * std::max(H, qd) * 4),
                 o_as = take(size_t(pad) * std::max(H, qd) / 8), o_a2 = take(size_t(pad) * F * 4),
                 o_as2 = take(size_t(pad) * F / 8), o_qkv = take(size_t(pad) * N * 4 * pq.splits),
                 o_y = take(size_t(pad) * H * 4 * std::max(po.splits, pd.splits)),
                 o_qh = take(size_t(rows) * qd * 2), o_ql = take(size_t(rows) * qd * 2),
                 o_qs = take(size_t(rows) * c.n_heads * 4),
                 o_part = take(size_t(std::max(zs_g, zs_l)) > 1
                                   ? size_t(c.n_kv_heads) * ((rows * G + 31u) / 32u) * std::max(zs_g, zs_l) * 32u * kPfRecord * 4
                                   : 0);
    if (int rc = reserve(off); rc != XP_OK) return rc;
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

PrefillEngine* prefill_engine_create(const xp_session* s) {
    PrefillEngine* p = new (std::nothrow) PrefillEngine;
    if (!p) {
        set_error(XP_E_NOMEM, "prefill: out of host memory");
        return nullptr;
    }
    p->owner = s;
    if (session_weights(s, &p->w) != XP_OK) {
        delete p;
        return nullptr;
    }
    const xp_config& c = p->w.cfg;
    const uint32_t G = c.n_kv_heads && c.n_heads % c.n_kv_heads == 0 ? c.n_heads / c.n_kv_heads : 0;
    const char* why = nullptr;
    if (c.scale_fmt != XP_SCALE_F16_QUAD && c.scale_fmt != XP_SCALE_BF16_QUAD) why = "takes fp16 or bf16 quad scales";
    else if (c.head_dim != 256u || (G != 1u && G != 2u && G != 4u)) why = "takes 1, 2 or 4 query heads of 256 dims per kv head";
    else if (c.hidden % 128u || c.ffn % 128u || c.hidden > 8192u) why = "takes hidden and ffn sizes that are multiples of 128";
    if (why) {
        prefill_engine_destroy(p);
        set_error(XP_E_ARG, "prefill: the batched path %s", why);
        return nullptr;
    }
    if (hipMalloc(reinterpret_cast<void**>(&p->d_ids), size_t(c.max_seq) * 4) != hipSuccess) {
        p->d_ids = nullptr;
        prefill_engine_destroy(p);
        set_error(XP_E_NOMEM, "prefill: device memory (%u token ids)", c.max_seq);
        return nullptr;
    }
    return p;
}

int prefill_engine_run(PrefillEngine* p, const uint32_t* ids, uint32_t n, uint32_t pos0, hipStream_t st) {
    p->st = st;
    // the weights as they are now: an embedding table may have been uploaded
    // since the last run
    if (int rc = session_weights(p->owner, &p->w); rc != XP_OK) return rc;
    XP_HIP(hipMemcpyAsync(p->d_ids, ids, size_t(n) * 4, hipMemcpyHostToDevice, st));
    uint32_t most = kPfMaxRows;
    for (uint32_t c0 = 0; c0 < n;) {
        const uint32_t rows = std::min(most, n - c0);
        const int rc = p->chunk(p->d_ids + c0, rows, pos0 + c0);
        if (rc == XP_E_NOMEM && rows > 64u) {
            most = rows / 2u;   // nothing of this chunk was queued: shorter ones
            clear_error();
            continue;
        }
        if (rc != XP_OK) {
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
    if (p->d_ids) (void)hipFree(p->d_ids);
    delete p;
}

}  // namespace xp
