// The prompt prefill's attention launch with plain arguments, for a test that
// measures its error by itself (through a session the GEMMs' and the cache's
// rounding cover it). Row records need splits >= 2.
#include "../../xpose_amd/csrc/xp_launch.hpp"

extern "C" int test_prefill_attention(void* qh, void* ql, float* qscale, uint16_t* kc, uint16_t* vc, uint32_t rows,
                                      uint32_t kv_heads, uint32_t group, uint32_t pos0, uint32_t window, float scale,
                                      void* a, float* asum, float* part, uint32_t splits) {
    xp::PfAttnArgs p{};
    p.qh = static_cast<const _Float16*>(qh);
    p.ql = static_cast<const _Float16*>(ql);
    p.qscale = qscale;
    p.kc = kc;
    p.vc = vc;
    p.rows = rows;
    p.kv_heads = kv_heads;
    p.pos0 = pos0;
    p.window = window;
    p.scale = scale;
    p.a = a;
    p.asum = asum;
    p.nblk = kv_heads * group * 8u;
    p.part = part;
    return xp::launch_pf_attn(p, group, splits, nullptr);
}

extern "C" uint32_t test_prefill_attention_record() { return xp::kPfRecord; }
