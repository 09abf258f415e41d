// Prompt prefill of a decode session: every layer of a chunk of up to
// kPfMaxRows prompt positions, as GEMMs on the matrix cores.
//
// A prompt of n tokens is 2 n FLOP a weight and one read of the weights. In
// passes of 16 positions the weights were read and every stage's latency was
// paid n / 16 times (68 us a token); here a chunk pays them once and is bound
// by the matrix cores. The arithmetic is the batched step's (xp_bmm_device.hpp):
// activations as two bf16 terms, nibbles widened to bf16 128 + n exactly, one
// v_mfma_f32_16x16x32_bf16 pair per 32-wide quantisation block with the bias
// correction -136 sum(hi + lo) as the accumulator's start value, every block's
// product scaled by its own weight scale in fp32.
//
// Stages of a layer: q|k|v GEMM, QK-norm + RoPE + KV append, attention, o GEMM,
// residual + norms, gate|up GEMM (GeGLU epilogue), down GEMM, residual + norms.
// A GEMM whose tiles would leave CUs idle is split along k; its splits are
// added, in order, by the stage that reads the result.
//
// The staged operand is kept in MFMA operand order (pf_stage), so a wave's
// operand is one contiguous KiB; asum holds each row's block sums.
#include "xp_bmm_device.hpp"
#include "xp_device.hpp"
#include "xp_launch.hpp"

#include <algorithm>
#include <cmath>

namespace xp {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Stages word c (8 elements) of block blk of a row, in the layout of the
// chunk's GEMMs. 16-row operand tiles: lane l of a block's operand holds row
// l % 16 and word l / 16, as stage_word. 32-row tiles (wide), for
// v_mfma_f32_32x32x16_bf16, whose two k steps a block take words (0, 2) and
// (1, 3): lane l of step kk holds row l % 32 and word 2 (l / 32) + kk, so that
// a weight lane's two words are adjacent. Slot s of a word is element s / 2 +
// 4 (s % 2), the order widen_nibbles gives the weights.
__device__ __forceinline__ void pf_stage(u32x4* A, float* asum, bool wide, uint32_t nblk, uint32_t row,
                                         uint32_t blk, uint32_t c, const float (&v)[8]) {
    uint32_t hi[8], lo[8];
    float sum = 0.0f;
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) {
        const float t = v[sl / 2 + 4 * (sl % 2)];
        hi[sl] = bf16_bits_rn(t);
        const float hf = __uint_as_float(hi[sl] << 16);
        lo[sl] = bf16_bits_rn(t - hf);
        sum += hf + __uint_as_float(lo[sl] << 16);
    }
    const uint32_t tr = wide ? 32u : 16u, rr = row % tr;
    const size_t tile = size_t(row / tr) * nblk + blk;
    u32x4* p = A + tile * (8u * tr) + (wide ? (c % 2u) * 128u + 32u * (c / 2u) : 16u * c) + rr;
    p[0] = u32x4{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16), hi[4] | (hi[5] << 16), hi[6] | (hi[7] << 16)};
    p[64] = u32x4{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16), lo[4] | (lo[5] << 16), lo[6] | (lo[7] << 16)};
    // the block's sum, from the four adjacent lanes that hold its words
    sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0xB1, 0xF, 0xF, false));
    sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x4E, 0xF, 0xF, false));
    if (c == 0) asum[tile * tr + rr] = sum;
}

// ---- residual add, norms and operand staging -------------------------------
// W waves a row (thread i of them takes the row's 8-element words i, i + 64 W,
// ...), RW rows a workgroup. Many rows: one wave a row, so every reduction
// stays in the wave, and 8 rows a workgroup, which writes whole 128-byte
// operand lines (16 left half of the CUs without one at 2000 rows: 15.0 us,
// 8: 12.5). Few rows: enough waves that a thread holds one word and has every
// split's share of it in flight at once.
//   tok set: x = embedding of tok[row]; stage rmsnorm(x) (1 + w_pre)
//   else:    x += rmsnorm(sum of the y splits) (1 + w_post), staged likewise
template <int NC, int RW, int W>
__global__ __launch_bounds__(RW * W * kWave) void pf_prep_kernel(PfPrepArgs a) {
    __shared__ float red[2][RW][W];
    const uint32_t rw = threadIdx.x / (W * kWave), th = threadIdx.x % (W * kWave);
    const uint32_t row = blockIdx.x * RW + rw;   // below rows_pad: whole workgroups of rows
    const uint32_t K = a.K, npair = K / 8;
    auto own = [&](int i) { return th + W * kWave * i < npair; };
    auto word = [&](int i) { return own(i) ? th + W * kWave * i : 0u; };
    auto row_sum = [&](float v, int slot) {
        v = wave_sum(v);
        if constexpr (W > 1) {
            if (th % kWave == 0) red[slot][rw][th / kWave] = v;
            __syncthreads();
            v = 0.0f;
#pragma unroll
            for (int w = 0; w < W; ++w) v += red[slot][rw][w];
        }
        return v;
    };
    float* x = a.x + size_t(row) * K;
    float xv[NC][8], wpre[NC][8];
    auto load_pre = [&]() {
#pragma unroll
        for (int i = 0; i < NC; ++i) ld8f(wpre[i], a.w_pre + 8 * word(i));
    };
    if constexpr (NC == 1) load_pre();   // with the rows; more words would spill
    if (a.tok) {
        uint32_t t = a.tok[min(row, a.rows - 1u)];
        if (t >= a.vocab) t = 0;
        const uint32_t nblk = K / kBlk;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const uint32_t p = word(i);
            if (a.etable) {
                ld8f(xv[i], a.etable + size_t(t) * K + 8 * p);
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[i][e] *= a.escale;
            } else {
                const uint32_t blk = p / 4u;
                const uint32_t wd =
                    static_cast<const uint32_t*>(a.ewq)[((size_t(t / kGrp) * nblk + blk) * kGrp + t % kGrp) * 4 + p % 4u];
                const uint16_t h = static_cast<const uint16_t*>(a.esc)[(size_t(blk / 4) * a.vocab + t) * 4 + blk % 4];
                const float sc = a.efmt == XP_SCALE_F16_QUAD ? f16_bits_to_f32(h) : __uint_as_float(uint32_t(h) << 16);
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[i][e] = (float(int((wd >> (4 * e)) & 15u) - 8) * sc) * a.escale;
            }
        }
    } else {
        float yv[NC][8], wpost[NC][8];
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            ld8f(xv[i], x + 8 * word(i));
            ld8f(wpost[i], a.w_post + 8 * word(i));
            ld8f(yv[i], a.y + size_t(row) * K + 8 * word(i));
        }
        // the further splits, in order, U of them in flight
        constexpr uint32_t U = NC == 1 ? 6 : 1;
        const size_t sst = size_t(a.rows_pad) * K;
        for (uint32_t s = 1; s < a.ysplit; s += U) {
            float t[U][NC][8];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < NC; ++i)
                    ld8f(t[u][i], a.y + min(s + u, a.ysplit - 1u) * sst + size_t(row) * K + 8 * word(i));
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                if (s + u >= a.ysplit) break;
#pragma unroll
                for (int i = 0; i < NC; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e) yv[i][e] += t[u][i][e];
            }
        }
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NC; ++i)
            if (own(i))
#pragma unroll
                for (int e = 0; e < 8; ++e) ss = fmaf(yv[i][e], yv[i][e], ss);
        const float post = rsq_hw(row_sum(ss, 0) / float(K) + a.eps);
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) xv[i][e] = xv[i][e] + yv[i][e] * post * (1.0f + wpost[i][e]);
    }
    float sx = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        if (!own(i)) continue;
        float4* xo = reinterpret_cast<float4*>(x + 8 * word(i));
        xo[0] = float4{xv[i][0], xv[i][1], xv[i][2], xv[i][3]};
        xo[1] = float4{xv[i][4], xv[i][5], xv[i][6], xv[i][7]};
#pragma unroll
        for (int e = 0; e < 8; ++e) sx = fmaf(xv[i][e], xv[i][e], sx);
    }
    if constexpr (NC > 1) load_pre();
    const float pre = rsq_hw(row_sum(sx, 1) / float(K) + a.eps);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const uint32_t p = word(i);
        if (!own(i)) continue;   // whole quads: K is a multiple of 128
        float w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = xv[i][e] * pre * (1.0f + wpre[i][e]);
        pf_stage(static_cast<u32x4*>(a.a), a.asum, a.wide, K / kBlk, row, p / 4u, p % 4u, w);
    }
}

// ---- int4 GEMM ---------------------------------------------------------------
// Workgroup: 128 rows x 128 columns (GE: 64 columns of gate and of up), four
// waves of 64 x 64, on v_mfma_f32_32x32x16_bf16 (the 16-row form lets no vector
// instruction issue beside it: 25 cycles for a 16-cycle multiply and three
// FMAs where the 32-row form takes 40 for 32 and six, measured; a block's
// scaling and nibble widening are about seven a multiply). Operand blocks
// pass through two LDS buffers: registers -> LDS for block i + 1 and global
// -> registers for block i + 3 are issued before block i's products, one
// barrier a block (with one block less in flight a lone workgroup on a CU
// waited out the load latency, 0.83 us, every block). Weights go straight to registers (each lane's two words of
// its column's KM4 block), three blocks ahead, scale quads one quad ahead.
// Workgroups are dealt to the XCDs in turn, so work item i of the launch goes
// to XCD i % 8: each XCD takes its own run of column tiles for every row
// tile, which keeps its weights and a few row tiles' operands in its L2.
template <int FMT, bool GE>
__global__ __launch_bounds__(256, 2) void pf_gemm_kernel(PfGemmArgs a) {
    constexpr uint32_t TM = 4;                            // 32-row tiles of the workgroup
    constexpr uint32_t STAGE = TM * 256u, R = STAGE / 256u;   // 16-byte words a block
    constexpr uint32_t HS = 68;                           // GE: floats a row of the output exchange
    constexpr uint32_t LDS_A = 2u * STAGE * 16u, LDS_C = 2u * 256u * 4u;
    constexpr uint32_t LDS_H = GE ? 128u * HS * 4u : 0u;
    constexpr uint32_t LDS = LDS_A + LDS_C > LDS_H ? LDS_A + LDS_C : LDS_H;
    __shared__ __attribute__((aligned(16))) unsigned char smem[LDS];
    u32x4* As = reinterpret_cast<u32x4*>(smem);
    float* Cs = reinterpret_cast<float*>(smem + LDS_A);

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const uint32_t wm = wave / 2u, wn = wave % 2u;
    const uint32_t c32 = lane % 32u, half = lane / 32u;
    // work item: XCD x owns columns [x nC / 8, (x + 1) nC / 8) of the nC =
    // splits x column tiles, rows outer, columns inner
    const uint32_t xcd = blockIdx.x % 8u, seq = blockIdx.x / 8u;
    const uint32_t nC = a.n_tiles * a.splits;
    const uint32_t c0 = xcd * nC / 8u, cn = (xcd + 1u) * nC / 8u - c0;
    if (cn == 0 || seq >= cn * a.m_wgs) return;
    const uint32_t c = c0 + seq % cn, bm = seq / cn;
    const uint32_t s = c / a.n_tiles, bn = c % a.n_tiles;
    const uint32_t nblk = a.nblk;
    const uint32_t q0 = s * a.qsplit, q1 = min(q0 + a.qsplit, nblk / 4u);
    const uint32_t kend = q1 * 4u, mt32 = (a.m_tiles + 1u) / 2u;

    // the wave's two 32-column tiles: tile t's matrix and column (uniform)
    rsrc_t rw[2], rs[2];
    uint32_t wo[2], so[2], sst[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        uint32_t ct, m = 0;                               // 32-column tile within its matrix, matrix
        if constexpr (GE) {
            ct = bn * 2u + wn;
            m = uint32_t(t);
        } else {
            ct = (bn * 2u + wn) * 2u + t;
#pragma unroll
            for (uint32_t i = 1; i < 3; ++i)
                if (i < a.n_mats && ct >= a.tile0[i] / 2u) m = i;
            ct -= a.tile0[m] / 2u;
        }
        const uint32_t cols = a.mats[m].cols;
        rw[t] = make_rsrc(a.mats[m].wq, cols * nblk * 16u);
        rs[t] = make_rsrc(a.mats[m].sc, cols * nblk * 2u);
        wo[t] = ((ct / 2u) * nblk * kGrp + (ct % 2u) * 32u) * 16u;
        so[t] = ct * 256u;
        sst[t] = cols * 8u;
    }
    const uint32_t wv = c32 * 16u + half * 8u, sv = c32 * 8u;
    // operand staging: 16-byte word i of a block = (row tile, word)
    const rsrc_t rA = make_rsrc(a.a, mt32 * nblk * 4096u), rC = make_rsrc(a.asum, mt32 * nblk * 128u);
    uint32_t ao[R];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) ao[r] = (min(bm * TM + r, mt32 - 1u) * nblk * 256u + tid) * 16u;
    // block sums: word tid of a block (threads past the 128 rows repeat rows
    // and store past them: no branch, which the compiler would sink the
    // loop's FMAs over)
    const uint32_t co = (min(bm * TM + (tid / 32u) % 4u, mt32 - 1u) * nblk * 32u + tid % 32u) * 4u;
    u32x4 ra[2][R];                                       // blocks in flight, by parity
    uint32_t rc[2];
    auto load_a = [&](uint32_t i, uint32_t kb) {
        kb = min(kb, kend - 1u);                          // past the end: the last block again, not used
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) ra[i][r] = __builtin_amdgcn_raw_buffer_load_b128(rA, int(ao[r]), int(kb * 4096u), 0);
        rc[i] = __builtin_amdgcn_raw_buffer_load_b32(rC, int(co), int(kb * 128u), 0);
    };
    auto store_a = [&](uint32_t i) {
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) As[i * STAGE + tid + r * 256u] = ra[i][r];
        Cs[i * 256u + tid] = -136.0f * __uint_as_float(rc[i]);
    };
    u32x2 w[4][2], sc[2][2];
    auto load_w = [&](u32x2 (&o)[2], uint32_t kb) {
        kb = min(kb, kend - 1u);
#pragma unroll
        for (int t = 0; t < 2; ++t) o[t] = __builtin_amdgcn_raw_buffer_load_b64(rw[t], int(wv), int(wo[t] + kb * 1024u), 0);
    };
    auto load_s = [&](u32x2 (&o)[2], uint32_t q) {
        q = min(q, q1 - 1u);
#pragma unroll
        for (int t = 0; t < 2; ++t) o[t] = __builtin_amdgcn_raw_buffer_load_b64(rs[t], int(sv), int(so[t] + q * sst[t]), 0);
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][t][r] = 0.0f;
    const NibConst nk = nib_const();

    load_a(0, q0 * 4u);
    load_s(sc[0], q0);
    load_w(w[0], q0 * 4u);
    load_a(1, q0 * 4u + 1u);
    load_w(w[1], q0 * 4u + 1u);
    load_w(w[2], q0 * 4u + 2u);
    store_a(0);
    load_a(0, q0 * 4u + 2u);
    for (uint32_t q = q0; q < q1; ++q) {
        load_s(sc[1], q + 1u);
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t buf = j % 2u;                  // a split starts and ends on a quad
            __syncthreads();
            // every wave is past the products of the block before, which
            // read the other buffer
            store_a(buf ^ 1u);
            load_a(buf ^ 1u, q * 4u + j + 3u);
            load_w(w[(j + 3u) % 4u], q * 4u + j + 3u);
            bf16x8 bw[2][2];
            float f[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                bw[t][0] = as_bf16x8(widen_nibbles(w[j][t].x, nk));
                bw[t][1] = as_bf16x8(widen_nibbles(w[j][t].y, nk));
                f[t] = quad_scale<FMT>(sc[0][t], j);
            }
            f32x16 p[2], pp[2];
            auto scale = [&](int m) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[m][t][r] = fmaf(f[t], pp[t][r], acc[m][t][r]);
            };
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const uint32_t b = wm * 2u + m;
                const u32x4* A = As + buf * STAGE + b * 256u + lane;
                f32x16 cr;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(&Cs[buf * 256u + b * 32u + 8u * i + 4u * half]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) cr[4 * i + r] = v[r];
                }
                const bf16x8 h0 = as_bf16x8(A[0]), l0 = as_bf16x8(A[64]), h1 = as_bf16x8(A[128]), l1 = as_bf16x8(A[192]);
                // both hi steps first: after them the correction has cancelled
                // and the lo terms are added at the result's magnitude
#pragma unroll
                for (int t = 0; t < 2; ++t) p[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h0, bw[t][0], cr, 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) p[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h1, bw[t][1], p[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) p[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l0, bw[t][0], p[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) p[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l1, bw[t][1], p[t], 0, 0, 0);
                if (m > 0) scale(m - 1);                  // tile 0 is scaled while tile 1 multiplies
#pragma unroll
                for (int t = 0; t < 2; ++t) pp[t] = p[t];
                __builtin_amdgcn_sched_barrier(0);
            }
            scale(1);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) sc[0][t] = sc[1][t];
    }
    // C layout: column lane % 32, rows 8 i + 4 (lane / 32) + r in word 4 i + r
    if constexpr (!GE) {
        float* out = a.out + size_t(s) * a.m_tiles * 16u * a.ldo;
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t row = (bm * TM + wm * 2u + m) * 32u + 8u * i + 4u * half;
                if (row >= a.m_tiles * 16u) continue;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        out[size_t(row + r) * a.ldo + ((bn * 2u + wn) * 2u + t) * 32u + c32] = acc[m][t][4 * i + r];
            }
    } else {
        // gelu(gate) up through LDS into the down GEMM's operand order
        float* H = reinterpret_cast<float*>(smem);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    H[((wm * 2u + m) * 32u + 8u * i + 4u * half + r) * HS + wn * 32u + c32] =
                        gelu_hw(acc[m][0][4 * i + r]) * acc[m][1][4 * i + r];
        __syncthreads();
        // 128 rows x 8 words, a block's four words in adjacent lanes
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t wd = tid + i * 256u, cw = wd % 4u, rr = (wd / 4u) % 32u, blk = (wd / 128u) % 2u, mt = wd / 256u;
            if (bm * TM + mt >= mt32) break;              // the whole workgroup
            float v[8];
            ld8f(v, H + (mt * 32u + rr) * HS + blk * 32u + cw * 8u);
            pf_stage(static_cast<u32x4*>(a.a_out), a.asum_out, true, a.nblk_out, (bm * TM + mt) * 32u + rr, bn * 2u + blk, cw, v);
        }
    }
}

// The GEMM for a few row tiles (a short prompt): latency, not the matrix
// cores, bounds it, so the eight waves of a workgroup split k instead of
// sharing operands through LDS. Wave w loads every operand of its next D
// blocks at once, straight in operand order, and the waves' tiles meet in LDS
// at the end, added in wave order. Workgroup: 16 MT rows x 16 T columns (GE:
// 32 columns of both matrices, T = 4).
template <int FMT, int MT, int T, int D, bool GE>
__global__ __launch_bounds__(512) void pf_gemm_small_kernel(PfGemmArgs a) {
    static_assert(!GE || T == 4, "two gate and two up tiles");
    constexpr int MR = MT * T > 8 ? 8 / T : MT;           // row tiles a reduction pass takes
    __shared__ f32x4 red[8][MR * T * 64];
    __shared__ __attribute__((aligned(16))) float hb[GE ? MR * 16 : 1][36];
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const uint32_t col16 = lane % 16u, wsel = lane / 16u;
    const uint32_t xcd = blockIdx.x % 8u, seq = blockIdx.x / 8u;
    const uint32_t nC = a.n_tiles * a.splits;
    const uint32_t c0 = xcd * nC / 8u, cn = (xcd + 1u) * nC / 8u - c0;
    if (cn == 0 || seq >= cn * a.m_wgs) return;
    const uint32_t c = c0 + seq % cn, bm = seq / cn;
    const uint32_t s = c / a.n_tiles, bn = c % a.n_tiles;
    const uint32_t nblk = a.nblk;
    const uint32_t s0 = s * a.qsplit * 4u, s1 = min(s0 + a.qsplit * 4u, nblk);
    const uint32_t kc = (s1 - s0 + 7u) / 8u;
    const uint32_t kb0 = min(s0 + wave * kc, s1), kb1 = min(kb0 + kc, s1);
    rsrc_t rw[T], rs[T];
    uint32_t wo[T], so[T], sst[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        uint32_t ct, m = 0;
        if constexpr (GE) {
            ct = bn * 2u + t % 2u;
            m = t / 2u;
        } else {
            ct = bn * T + t;
#pragma unroll
            for (uint32_t i = 1; i < 3; ++i)
                if (i < a.n_mats && ct >= a.tile0[i]) m = i;
            ct -= a.tile0[m];
        }
        const uint32_t cols = a.mats[m].cols;
        rw[t] = make_rsrc(a.mats[m].wq, cols * nblk * 16u);
        rs[t] = make_rsrc(a.mats[m].sc, cols * nblk * 2u);
        wo[t] = ((ct / 4u) * nblk * kGrp + (ct % 4u) * 16u) * 16u;
        so[t] = ct * 128u;
        sst[t] = cols * 8u;
    }
    const rsrc_t rA = make_rsrc(a.a, a.m_tiles * nblk * 2048u), rC = make_rsrc(a.asum, a.m_tiles * nblk * 64u);
    struct Ops {
        u32x4 hi[MT], lo[MT];
        uint32_t as[MT];   // lane l's word of the block sums, row 4 (l / 16) + l % 4
        uint32_t w[T];
    };
    auto load = [&](Ops& o, uint32_t blk) {
#pragma unroll
        for (int t = 0; t < T; ++t)
            o.w[t] = __builtin_amdgcn_raw_buffer_load_b32(rw[t], int(col16 * 16u + wsel * 4u), int(wo[t] + blk * 1024u), 0);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const uint32_t mb = min(bm * MT + m, a.m_tiles - 1u) * nblk + blk;
            o.hi[m] = __builtin_amdgcn_raw_buffer_load_b128(rA, int(lane * 16u), int(mb * 2048u), 0);
            o.lo[m] = __builtin_amdgcn_raw_buffer_load_b128(rA, int(lane * 16u + 1024u), int(mb * 2048u), 0);
            o.as[m] = __builtin_amdgcn_raw_buffer_load_b32(rC, int(wsel * 16u + (lane % 4u) * 4u), int(mb * 64u), 0);
        }
    };
    const NibConst nk = nib_const();
    f32x4 acc[MT][T];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[m][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t k = kb0; k < kb1; k += D) {
        // D <= 5 consecutive blocks lie in at most two scale quads
        const uint32_t q0 = k / 4u;
        u32x2 sc[2][T];
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < T; ++t)
                sc[i][t] = __builtin_amdgcn_raw_buffer_load_b64(rs[t], int(col16 * 8u), int(so[t] + min(q0 + i, nblk / 4u - 1u) * sst[t]), 0);
        Ops ops[D];
#pragma unroll
        for (int j = 0; j < D; ++j) {
            load(ops[j], min(k + j, kb1 - 1u));           // past the end: the last block again, not used
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (k + j >= kb1) break;
            Ops& o = ops[j];
            f32x4 cr[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m)
                cr[m] = f32x4{-nk.bias * dpp_quad_bcast<0>(o.as[m]), -nk.bias * dpp_quad_bcast<1>(o.as[m]),
                              -nk.bias * dpp_quad_bcast<2>(o.as[m]), -nk.bias * dpp_quad_bcast<3>(o.as[m])};
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const bf16x8 bw = as_bf16x8(widen_nibbles(o.w[t], nk));
                const float f = quad_scale<FMT>((k + j) / 4u != q0 ? sc[1][t] : sc[0][t], (k + j) % 4u);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    f32x4 p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(o.hi[m]), bw, cr[m], 0, 0, 0);
                    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(o.lo[m]), bw, p, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[m][t][r] = fmaf(f, p[r], acc[m][t][r]);
                }
            }
        }
    }
#pragma unroll
    for (int m0 = 0; m0 < MT; m0 += MR) {
        if (m0 > 0) __syncthreads();
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int t = 0; t < T; ++t) red[wave][(m * T + t) * 64 + lane] = acc[m0 + m][t];
        __syncthreads();
        auto total = [&](uint32_t i) {
            f32x4 v = red[0][i];
#pragma unroll
            for (int w = 1; w < 8; ++w) v += red[w][i];
            return v;
        };
        if constexpr (!GE) {
            float* out = a.out + size_t(s) * a.m_tiles * 16u * a.ldo;
#pragma unroll
            for (uint32_t i0 = 0; i0 < MR * T * 64u; i0 += 512u) {
                const uint32_t i = i0 + tid, t = (i / 64u) % T, mt = bm * MT + m0 + i / (64u * T);
                if (i >= MR * T * 64u || mt >= a.m_tiles) break;   // whole waves
                const f32x4 v = total(i);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    out[size_t(mt * 16u + 4u * wsel + r) * a.ldo + (bn * T + t) * 16u + col16] = v[r];
            }
        } else {
            // gate tile t at (m 4 + t), its up tile at (m 4 + t + 2)
            static_assert(MR * 2 * 64 <= 512, "one gate tile word a thread");
            if (tid < MR * 128u) {
                const uint32_t m = tid / 128u, t = (tid / 64u) % 2u;
                const f32x4 g = total((m * 4u + t) * 64u + lane), u = total((m * 4u + t + 2u) * 64u + lane);
#pragma unroll
                for (int r = 0; r < 4; ++r) hb[m * 16u + 4u * wsel + r][t * 16u + col16] = gelu_hw(g[r]) * u[r];
            }
            __syncthreads();
            const uint32_t m = tid / 64u, mt = bm * MT + m0 + m;   // 64 words a row tile: whole waves
            if (m < MR && mt < a.m_tiles) {
                float v[8];
                ld8f(v, &hb[m * 16u + (tid / 4u) % 16u][8u * (tid % 4u)]);
                pf_stage(static_cast<u32x4*>(a.a_out), a.asum_out, false, a.nblk_out, mt * 16u + (tid / 4u) % 16u, bn, tid % 4u, v);
            }
        }
    }
}

// ---- QK-norm, RoPE, KV append ----------------------------------------------
// One wave per (row, head): lane l holds dims 2 l, 2 l + 1 and the same plus
// 128 (its RoPE pairs). Query rows go out as two fp16 terms of q 2^e, e per
// row such that the largest magnitude is in [2^13, 2^14) (22 bits of every
// element within 2^-39 of the largest), with 2^-e in qscale; keys and values
// to the cache.
__global__ __launch_bounds__(256) void pf_qk_kernel(PfQkArgs a, RopeFreq f) {
    const uint32_t slots = a.n_heads + 2u * a.kv_heads;
    const uint32_t w = blockIdx.x * 4u + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint32_t row = w / slots, h = w % slots;
    if (row >= a.rows) return;
    const uint32_t N = slots * 256u, pos = a.pos0 + row;
    float2 lo{0.0f, 0.0f}, hi{0.0f, 0.0f};
    for (uint32_t s = 0; s < a.splits; ++s) {
        const float* p = a.qkv + (size_t(s) * a.rows_pad + row) * N + h * 256u + 2u * lane;
        const float2 u = *reinterpret_cast<const float2*>(p), v = *reinterpret_cast<const float2*>(p + 128);
        lo.x += u.x; lo.y += u.y; hi.x += v.x; hi.y += v.y;
    }
    const bool is_q = h < a.n_heads;
    if (h >= a.n_heads + a.kv_heads) {
        uint16_t* o = a.vc + (size_t(pos) * a.kv_heads + (h - a.n_heads - a.kv_heads)) * 256u + 2u * lane;
        *reinterpret_cast<uint32_t*>(o) = uint32_t(f32_to_f16_bits(lo.x)) | (uint32_t(f32_to_f16_bits(lo.y)) << 16);
        *reinterpret_cast<uint32_t*>(o + 128) = uint32_t(f32_to_f16_bits(hi.x)) | (uint32_t(f32_to_f16_bits(hi.y)) << 16);
        return;
    }
    const float* nw = is_q ? a.qw : a.kw;
    const float2 wl = *reinterpret_cast<const float2*>(nw + 2u * lane), wh = *reinterpret_cast<const float2*>(nw + 128 + 2u * lane);
    const float ss = wave_sum(fmaf(lo.x, lo.x, fmaf(lo.y, lo.y, fmaf(hi.x, hi.x, hi.y * hi.y))));
    const float sc = rsq_hw(ss / 256.0f + a.eps);
    float l0 = lo.x * sc * (1.0f + wl.x), l1 = lo.y * sc * (1.0f + wl.y);
    float h0 = hi.x * sc * (1.0f + wh.x), h1 = hi.y * sc * (1.0f + wh.y);
    auto rot = [&](float& p, float& q, float inv) {
        float sn, cs;
        sincosf(float(pos) * inv, &sn, &cs);
        const float t = p * cs - q * sn;
        q = q * cs + p * sn;
        p = t;
    };
    rot(l0, h0, f.inv[2u * lane]);
    rot(l1, h1, f.inv[2u * lane + 1u]);
    if (!is_q) {
        uint16_t* o = a.kc + (size_t(pos) * a.kv_heads + (h - a.n_heads)) * 256u + 2u * lane;
        *reinterpret_cast<uint32_t*>(o) = uint32_t(f32_to_f16_bits(l0)) | (uint32_t(f32_to_f16_bits(l1)) << 16);
        *reinterpret_cast<uint32_t*>(o + 128) = uint32_t(f32_to_f16_bits(h0)) | (uint32_t(f32_to_f16_bits(h1)) << 16);
        return;
    }
    const float m = wave_max(fmaxf(fmaxf(fabsf(l0), fabsf(l1)), fmaxf(fabsf(h0), fabsf(h1))));
    // 2^e from the exponent field of the largest magnitude (biased ex: the
    // magnitude is in [2^(ex - 127), 2^(ex - 126))); zero and infinite rows,
    // and those below 2^-111 (whose scores are zero in fp32 sums), take e = 0
    const uint32_t ex = (__float_as_uint(m) >> 23) & 255u;
    const float up = ex >= 16u && ex <= 254u ? __uint_as_float((267u - ex) << 23) : 1.0f;
    const float down = 1.0f / up;
    const uint32_t g = a.n_heads / a.kv_heads, kvh = h / g, hg = h % g;
    const size_t qr = (size_t(kvh) * a.rows + row) * g + hg;
    auto put = [&](float u, float v, uint32_t d) {
        u *= up;
        v *= up;
        const _Float16 uh = _Float16(u), vh = _Float16(v);
        const f16x2 hh{uh, vh}, ll{_Float16(u - float(uh)), _Float16(v - float(vh))};
        *reinterpret_cast<f16x2*>(a.qh + qr * 256u + d) = hh;
        *reinterpret_cast<f16x2*>(a.ql + qr * 256u + d) = ll;
    };
    put(l0, l1, 2u * lane);
    put(h0, h1, 128u + 2u * lane);
    if (lane == 0) a.qscale[qr] = down;
}

// ---- attention ----------------------------------------------------------------
// Workgroup: 32 query rows (32 / G consecutive positions of one kv head's G
// query heads) over the keys they may see, 128 at a time through LDS; wave w
// takes rows 16 (w % 2) .. and keys 32 (w / 2) .. of each 128. Scores are
// formed transposed, S^T = K Q^T, so a lane holds four consecutive keys of one
// query per 16-key tile: with the keys of a 32-key step taken in the order
// (4 g + 0..3, 16 + 4 g + 0..3) for lane group g, those are exactly the lane's
// operand words of O^T = V^T P^T, and P never leaves its lane. V is transposed
// into LDS in that key order while it is staged (8 keys x 8 dims a thread).
// K and V are fp16 as the cache holds them. q and p are two fp16 terms each
// (22 bits), which costs accuracy that the sums win back: the matrix units round
// at the running sum's size several times an instruction, so scores are formed
// over 64 dims at a time, low terms first, and the values of a step on their own,
// and both are added in fp32; the exponent is one fused multiply-add of the
// score. Distance from float64 of the same q and cache, against the token steps'
// attention (fp32 q and p) on the same rows: 32 rows 8.9e-8 (9.3e-8), 2000 rows
// 1.36e-7 (1.40e-7), in a window of 512 1.40e-7 (1.45e-7), from position 1500
// 1.88e-7 (1.84e-7); with one chain a score and a value 1.28 to 1.79 times the
// steps'. It takes the same time (2000 tokens 8.71 ms, 300 3.72). Two waves a SIMD (a lone wave issues a vector instruction
// every 8 cycles), cache rows through raw buffers, one descriptor a load that
// starts at the load's first row (scalar arithmetic only) and ends at the last
// key: rows past it read as zeros.
//
// A masked key has weight 0, which the value product would turn into NaN where
// its value is not finite. The keys that only some rows see (edge keys: up to
// 31 ahead of the first row and 31 that have left the last row's window) are
// looked at while their tile is staged: a non-finite value goes to LDS as
// zero, the key's bit is set, and the rows that do see the key become NaN at
// the end (all of a row: the o product mixes its dims). A wave looks only where
// its 32 keys of a tile hold edge keys, which costs nothing that shows: 300 tokens
// of 26 layers 3.55 ms with it and without, 2000 tokens 8.83-8.90 and 8.82-8.88.
constexpr uint32_t kPaThreads = 512, kPaKeys = 128;
constexpr float kPaPScale = 16384.0f;   // p 2^14: the low term keeps bits to 2^-38

struct __attribute__((aligned(16))) PaSmem {   // 16-byte LDS accesses
    union {
        struct {
            unsigned char k[kPaKeys * 512];     // key row, 16-byte word w at w ^ (key & 7)
            unsigned char v[256 * kPaKeys * 2]; // dim row of 16 key chunks, chunk c at c ^ pa_swz(dim)
        } t;
        struct {
            float o[4][32][260];                // each key group's sums
            float m[4][32], l[4][32];
        } c;
    };
    uint32_t bad[2];   // non-finite edge keys: that have left a window, that lie ahead
};
// Chunk swizzle of V's dim rows: distinct over 8 consecutive dims (a read's
// lanes) and over dims 8 apart (a transposing write's lanes).
__device__ __forceinline__ uint32_t pa_swz(uint32_t dim) { return (dim ^ (dim >> 3)) & 7u; }

template <int G>
__global__ __launch_bounds__(kPaThreads) void pf_attn_kernel(PfAttnArgs a) {
    __shared__ PaSmem sm;
    constexpr uint32_t TOK = 32u / G;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const uint32_t rg = wave % 2u, kg = wave / 2u, n16 = lane % 16u, g = lane / 16u;
    const uint32_t kvh = blockIdx.y, z = blockIdx.z, nz = gridDim.z;
    const uint32_t t0 = (gridDim.x - 1u - blockIdx.x) * TOK;          // the longest spans first
    const uint32_t tl = min(t0 + TOK, a.rows) - 1u;                    // last position of the workgroup
    const uint32_t last = a.pos0 + tl, first = a.pos0 + t0;
    uint32_t k0 = a.window && first + 1u > a.window ? first + 1u - a.window : 0u;
    uint32_t kn = last + 1u;                                           // keys [k0, kn)
    const uint32_t low = k0;
    // keys every row of the workgroup sees: no mask between the two
    const uint32_t free0 = a.window && last + 1u > a.window ? last + 1u - a.window : 0u;
    if (nz > 1u) {                                                     // this workgroup's share of the tiles
        const uint32_t tiles = (kn - k0 + kPaKeys - 1u) / kPaKeys, per = (tiles + nz - 1u) / nz;
        k0 += min(z * per, tiles) * kPaKeys;
        kn = min(kn, k0 + per * kPaKeys);
    }
    const uint32_t rowb = a.kv_heads * 512u;                           // bytes between cache rows
    const uint32_t kvbytes = (last + 1u) * rowb;
    auto rows_from = [&](const uint16_t* base, uint32_t row) {
        const uint32_t off = __builtin_amdgcn_readfirstlane(min(row * rowb, kvbytes));
        return make_rsrc(reinterpret_cast<const unsigned char*>(base) + off, __builtin_amdgcn_readfirstlane(kvbytes - off));
    };
    // K: 16-byte word i of the tile = key i / 32, word i % 32. V: thread's key
    // chunk tid / 32 = (32-key step, group) and dims 8 (tid % 32) ..
    const uint32_t ko = (tid / 32u) * rowb + kvh * 512u + (tid % 32u) * 16u;
    const uint32_t vch = tid / 32u, vd = tid % 32u;
    const uint32_t vo = ((vch / 4u) * 32u + (vch % 4u) * 4u) * rowb + kvh * 512u + vd * 16u;
    u32x4 kr[8], vr[8];
    auto load = [&](uint32_t kt) {
#pragma unroll
        for (uint32_t r = 0; r < 8; ++r)
            kr[r] = __builtin_amdgcn_raw_buffer_load_b128(rows_from(a.kc, kt + 16u * r), int(ko), 0, 0);
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j)
            vr[j] = __builtin_amdgcn_raw_buffer_load_b128(rows_from(a.vc, kt + (j & 3u) + (j >> 2) * 16u), int(vo), 0, 0);
    };
    auto store = [&](uint32_t kt) {
        const uint32_t ks = kt + (wave / 2u) * 32u;   // the wave's keys
        if (ks <= last && (ks < free0 || ks + 31u > first)) {
            // both halves of a word at once: an exponent of all ones carries into bit 15
            uint32_t any = 0;
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j)
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) any |= (vr[j][i] & 0x7C007C00u) + 0x04000400u;
            if (any & 0x80008000u) {
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) {
                    const uint32_t key = ks + (vch % 4u) * 4u + (j & 3u) + (j >> 2) * 16u;
                    const bool left = key < free0;
                    if (!left && key <= first) continue;
                    bool hit = false;
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        const uint32_t w = vr[j][i];
                        const uint32_t keep = ((w & 0x7C00u) != 0x7C00u ? 0xFFFFu : 0u) | ((w & 0x7C000000u) != 0x7C000000u ? 0xFFFF0000u : 0u);
                        hit |= keep != 0xFFFFFFFFu;
                        vr[j][i] = w & keep;
                    }
                    if (hit) atomicOr(&sm.bad[left ? 0 : 1], 1u << (left ? key - low : key - first - 1u));
                }
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < 8; ++r) {
            const uint32_t key = tid / 32u + 16u * r;
            *reinterpret_cast<u32x4*>(sm.t.k + key * 512u + ((tid % 32u) ^ (key & 7u)) * 16u) = kr[r];
        }
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {       // dim 8 vd + i of the eight keys
            u32x4 o;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                o[j] = __builtin_amdgcn_perm(vr[2 * j + 1][i / 2], vr[2 * j][i / 2], i % 2 ? 0x07060302u : 0x05040100u);
            const uint32_t dim = 8u * vd + i;
            *reinterpret_cast<u32x4*>(sm.t.v + dim * (kPaKeys * 2u) + (vch ^ pa_swz(dim)) * 16u) = o;
        }
    };
    if (k0 < kn) load(k0);
    if (tid < 2u) sm.bad[tid] = 0u;              // before the loop's first barrier
    // this lane's query row
    const uint32_t qi = rg * 16u + n16, tok = min(t0 + qi / G, a.rows - 1u);
    const uint32_t qpos = a.pos0 + tok;
    const uint32_t qlow = a.window && qpos + 1u > a.window ? qpos + 1u - a.window : 0u;
    const size_t qr = (size_t(kvh) * a.rows + tok) * G + qi % G;
    f16x8 qh[8], ql[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        qh[s] = *reinterpret_cast<const f16x8*>(a.qh + qr * 256u + s * 32 + g * 8u);
        ql[s] = *reinterpret_cast<const f16x8*>(a.ql + qr * 256u + s * 32 + g * 8u);
    }
    const float qs = a.qscale[qr] * a.scale * 1.4426950408889634f;
    const uint32_t free1 = min(first + 1u, kn);
    // read offsets: the swizzles repeat every 2 steps of 32 dims of K and every
    // 4 value tiles, the rest are constants
    uint32_t ka[2], va[4];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) ka[i] = (kg * 32u + n16) * 512u + ((4u * i + g) ^ (n16 & 7u)) * 16u;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) va[i] = (16u * i + n16) * (kPaKeys * 2u) + ((kg * 4u + g) ^ pa_swz(16u * i + n16)) * 16u;
    f32x4 o[16];
#pragma unroll
    for (int d = 0; d < 16; ++d) o[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;
    for (uint32_t kt = k0; kt < kn; kt += kPaKeys) {
        __syncthreads();                         // the tile before has been read by every wave
        store(kt);
        __syncthreads();
        if (kt + kPaKeys < kn) load(kt + kPaKeys);
        const uint32_t kk = kt + kg * 32u;       // this wave's keys
        if (kk >= kn) continue;
        // 64 dims at a time, low terms first, added in fp32 pairwise: fewer
        // roundings at the sum's size than in one chain
        f32x4 st[2], part[2];
#pragma unroll
        for (int s = 0; s < 8; s += 2)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f16x8 kv[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) kv[i] = *reinterpret_cast<const f16x8*>(sm.t.k + ka[i] + 16u * 512u * t + 64u * s);
                f32x4 h{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 2; ++i) h = __builtin_amdgcn_mfma_f32_16x16x32_f16(kv[i], ql[s + i], h, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 2; ++i) h = __builtin_amdgcn_mfma_f32_16x16x32_f16(kv[i], qh[s + i], h, 0, 0, 0);
                if (s == 0) st[t] = h;
                else if (s == 2) st[t] += h;
                else if (s == 4) part[t] = h;
                else st[t] += part[t] + h;
            }
        if (kk < free0 || kk + 32u > free1) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t key = kk + t * 16 + 4u * g + r;
                    if (key > qpos || key < qlow || key >= kn) st[t][r] = -INFINITY;
                }
        }
        float mx = fmaxf(fmaxf(fmaxf(st[0][0], st[0][1]), fmaxf(st[0][2], st[0][3])),
                         fmaxf(fmaxf(st[1][0], st[1][1]), fmaxf(st[1][2], st[1][3]))) * qs;
        mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
        mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
        const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.0f : mn;
        const float alpha = __builtin_amdgcn_exp2f(m - ms);   // 0 on the first keys
        m = mn;
        f16x8 ph, pl;
        float ps = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(fmaf(st[t][r], qs, -ms)) * kPaPScale;
                ps += p;
                const _Float16 h = _Float16(p);
                ph[4 * t + r] = h;
                pl[4 * t + r] = _Float16(p - float(h));
            }
        l = l * alpha + ps;
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
            for (int d = 0; d < 16; ++d) o[d] *= alpha;
        }
        // a step's sum is formed by itself and added in one rounding: four a
        // step at the running sum's size, as one chain, round twice as much
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            const f16x8 vv = *reinterpret_cast<const f16x8*>(sm.t.v + va[d % 4] + 64u * (kPaKeys * 2u) * (d / 4));
            f32x4 x = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv, pl, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv, ph, x, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[d][r] += x[r];
            if (d % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // more reads ahead would spill
        }
    }
    // the row's sum over its four lane groups (each holds other keys)
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    // the key groups meet: every thread combines its own words of the rows
    __syncthreads();
    if (g == 0) {
        sm.c.m[kg][qi] = m;
        sm.c.l[kg][qi] = l;
    }
#pragma unroll
    for (int d = 0; d < 16; ++d) *reinterpret_cast<f32x4*>(&sm.c.o[kg][qi][16 * d + 4 * g]) = o[d];
    __syncthreads();
    // 32 rows x 32 words of 8 dims
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t w = tid + kPaThreads * i, r = w / 32u, c = w % 32u, t = t0 + r / G;
        float f[4], M = sm.c.m[0][r], L = 0.0f;
#pragma unroll
        for (int q = 1; q < 4; ++q) M = fmaxf(M, sm.c.m[q][r]);
        const float Ms = M == -INFINITY ? 0.0f : M;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f[q] = __builtin_amdgcn_exp2f(sm.c.m[q][r] - Ms);
            L += sm.c.l[q][r] * f[q];
        }
        float inv = nz > 1u ? 1.0f : 1.0f / L;
        if (sm.bad[0] | sm.bad[1]) {             // the row's first key and the keys ahead of the first row that it sees
            const uint32_t p = a.pos0 + t, lo = a.window && p + 1u > a.window ? p + 1u - a.window : 0u;
            auto from = [&](uint32_t base) { return lo <= base ? ~0u : lo - base < 32u ? ~0u << (lo - base) : 0u; };
            auto upto = [&](uint32_t base) { return p < base ? 0u : p - base < 31u ? (2u << (p - base)) - 1u : ~0u; };
            if ((sm.bad[0] & from(low) & upto(low)) | (sm.bad[1] & from(first + 1u) & upto(first + 1u))) inv = NAN;
        }
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float e[8];
            ld8f(e, &sm.c.o[q][r][8u * c]);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = fmaf(e[j], f[q] * inv, v[j]);
        }
        if (nz > 1u) {
            // record [workgroup][z][32 rows][4 + 256]: max, sum, unnormalised row
            float* rec = a.part + (((size_t(kvh) * gridDim.x + (t0 / TOK)) * nz + z) * 32u + r) * kPfRecord;
            *reinterpret_cast<float4*>(rec + 4u + 8u * c) = float4{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<float4*>(rec + 8u + 8u * c) = float4{v[4], v[5], v[6], v[7]};
            if (c == 0) {
                rec[0] = M;
                rec[1] = L;
            }
        } else if (t < a.rows) {                 // a row's lanes together
            const uint32_t k = (kvh * G + r % G) * 256u + 8u * c;
            pf_stage(static_cast<u32x4*>(a.a), a.asum, a.wide, a.nblk, t, k / 32u, c % 4u, v);
        }
    }
}

// Adds the records of a key-split attention (same grid without z), in split
// order, and stages the rows.
template <int G>
__global__ __launch_bounds__(256) void pf_attn_combine_kernel(PfAttnArgs a, uint32_t nz) {
    constexpr uint32_t TOK = 32u / G;
    const uint32_t tid = threadIdx.x, kvh = blockIdx.y, t0 = blockIdx.x * TOK;
    const float* rec = a.part + (size_t(kvh) * gridDim.x + blockIdx.x) * nz * (32u * kPfRecord);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t w = tid + 256u * i, r = w / 32u, c = w % 32u, t = t0 + r / G;
        if (t >= a.rows) continue;
        float M = -INFINITY;
        for (uint32_t z = 0; z < nz; ++z) M = fmaxf(M, rec[(size_t(z) * 32u + r) * kPfRecord]);
        float L = 0.0f, v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t z = 0; z < nz; ++z) {
            const float* p = rec + (size_t(z) * 32u + r) * kPfRecord;
            const float f = p[0] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(p[0] - M);
            L += f * p[1];
            float e[8];
            ld8f(e, p + 4u + 8u * c);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += f * e[j];
        }
        const float inv = 1.0f / L;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= inv;
        const uint32_t k = (kvh * G + r % G) * 256u + 8u * c;
        pf_stage(static_cast<u32x4*>(a.a), a.asum, a.wide, a.nblk, t, k / 32u, c % 4u, v);
    }
}

// Rows up to which the small kernel is used: one workgroup of row tiles. With
// the small / the 128-row kernel, 26 layers of hidden 1152: 33 rows 2.03 / 2.53
// ms, 64 2.16 / 2.54, 65 (two workgroups of row tiles) 2.64 / 2.57; 12 layers of
// 2048: 64 1.35 / 1.58, 65 1.66 / 1.61. Hidden 512 would gain up to 128 rows
// (0.87 / 0.99 ms).
constexpr uint32_t kPfSmallRows = 64;
// Blocks of k that a wave of the small kernel takes at once (its GeGLU form with
// four row tiles three, which is 245 of 256 registers), and its waves.
constexpr uint32_t kPfSmallD = 5, kPfSmallWaves = 8;
// Columns a GEMM workgroup takes: of the output, or (GeGLU) of each of the two matrices.
uint32_t pf_gemm_cols(int shape, bool geglu) {
    return geglu ? (shape == 2 ? 64u : 32u) : (shape == 2 ? 128u : 16u);
}

int launched(const char* who) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(XP_E_HIP, "%s: launch -> %s", who, hipGetErrorString(e));
    return XP_OK;
}

}  // namespace

int launch_pf_prep(const PfPrepArgs& a, hipStream_t st) {
    // x is updated in place, so no row may be taken twice: rows_pad is whole
    // operand tiles of 16 rows, which every RW below divides
    if (a.K % 128u || a.K > 8192u || a.rows_pad % 16u) return set_error(XP_E_ARG, "prefill staging: K=%u rows=%u", a.K, a.rows_pad);
#define XP_PREP(NC, RW, W) \
    hipLaunchKernelGGL((pf_prep_kernel<NC, RW, W>), dim3(a.rows_pad / RW), dim3(RW * W * kWave), 0, st, a)
    // A word a thread for up to 512 rows (26 layers of hidden 1152, 256 rows 2.84
    // against 3.00 ms, 320 3.56 against 3.73, 512 3.74 against 3.83), then a wave a
    // row; wider rows always, in as many waves as they have words for (12 layers of
    // 2048 in 4 waves: 32 rows 1.07 ms, 2000 6.75; in 16, of which 12 idle, 1.08, 6.82).
    if (a.K <= 1536u) {
        if (a.rows_pad <= 512u) XP_PREP(1, 1, 3);
        else XP_PREP(3, 8, 1);
    } else if (a.K <= 2048u) {
        XP_PREP(1, 1, 4);
    } else if (a.K <= 4096u) {
        XP_PREP(1, 1, 8);
    } else {
        XP_PREP(1, 1, 16);
    }
#undef XP_PREP
    return launched("prefill staging");
}

// Tile shapes by rows: few rows are latency-bound (the small kernel, two or
// four row tiles a workgroup), many are bound by the matrix cores (128 x
// 128 tiles, which read LDS least per product).
PfGemmPlan plan_pf_gemm(uint32_t rows, uint32_t cols, uint32_t nblk, bool geglu, int n_cu) {
    PfGemmPlan p{};
    const uint32_t mt = (rows + 15u) / 16u, nq = nblk / 4u;
    p.shape = mt <= 2u ? 0 : rows <= kPfSmallRows ? 1 : 2;
    const uint32_t bm = 2u << p.shape;
    const uint32_t bn = pf_gemm_cols(p.shape, geglu);
    p.m_wgs = (mt + bm - 1u) / bm;
    p.n_tiles = (cols + bn - 1u) / bn;
    p.splits = 1;
    p.qsplit = nq;
    if (geglu) return p;
    const uint32_t tiles = p.m_wgs * p.n_tiles, cu = uint32_t(n_cu > 0 ? n_cu : 256);
    if (p.shape < 2) {
        // as many quads a split as keep the waves at the blocks they take at
        // once, unless the CUs would be over-subscribed twice. One quad less a
        // split: 12 layers of hidden 2560, ffn 10240 1.45 against 1.42 ms for 32
        // rows, 1.93 against 1.88 for 64; of 1280, 5120 0.90 against 0.91, 1.11
        // against 1.13; of 512, 1152 and 2048 the same.
        const uint32_t per = std::max(kPfSmallWaves * kPfSmallD / 4u, (nq * tiles + 2u * cu - 1u) / (2u * cu));
        p.splits = (nq + per - 1u) / per;
        p.qsplit = (nq + p.splits - 1u) / p.splits;
        p.splits = (nq + p.qsplit - 1u) / p.qsplit;
        return p;
    }
    // Estimated time in us of `real` runs of `per` quads: a block takes 0.8 us
    // in a workgroup alone on its CU, 0.6 us a workgroup where two share one
    // (measured at 128 to 2000 rows), starting and ending one 3 and 1.5 us;
    // the partials move at about 5 TB/s out and back in.
    double best = 1e30;
    for (uint32_t s = 1; s <= nq; ++s) {
        const uint32_t per = (nq + s - 1u) / s, real = (nq + per - 1u) / per, each = (tiles * real + cu - 1u) / cu;
        const double t = (each == 1u ? 3.2 * per + 3.0 : each * (2.4 * per + 1.5)) + 8.0 / 5e6 * double(real) * rows * cols;
        if (t < best) {
            best = t;
            p.splits = real;
            p.qsplit = per;
        }
    }
    return p;
}

template <int FMT>
static void gemm_launch(const PfGemmArgs& a, int shape, bool ge, hipStream_t st) {
    const uint32_t nC = a.n_tiles * a.splits;
    const dim3 grid(8u * a.m_wgs * ((nC + 7u) / 8u)), blk(shape == 2 ? 256 : 512);
    if (ge) {
        if (shape == 0) hipLaunchKernelGGL((pf_gemm_small_kernel<FMT, 2, 4, int(kPfSmallD), true>), grid, blk, 0, st, a);
        else if (shape == 1) hipLaunchKernelGGL((pf_gemm_small_kernel<FMT, 4, 4, 3, true>), grid, blk, 0, st, a);
        else hipLaunchKernelGGL((pf_gemm_kernel<FMT, true>), grid, blk, 0, st, a);
    } else {
        if (shape == 0) hipLaunchKernelGGL((pf_gemm_small_kernel<FMT, 2, 1, int(kPfSmallD), false>), grid, blk, 0, st, a);
        else if (shape == 1) hipLaunchKernelGGL((pf_gemm_small_kernel<FMT, 4, 1, int(kPfSmallD), false>), grid, blk, 0, st, a);
        else hipLaunchKernelGGL((pf_gemm_kernel<FMT, false>), grid, blk, 0, st, a);
    }
}

int launch_pf_gemm(PfGemmArgs a, const PfGemmPlan& p, int fmt, bool geglu, hipStream_t st, const char* who) {
    a.m_wgs = p.m_wgs;
    a.n_tiles = p.n_tiles;
    a.splits = p.splits;
    a.qsplit = p.qsplit;
    const uint32_t bn = pf_gemm_cols(p.shape, geglu);
    uint32_t cols = 0;
    for (uint32_t i = 0; i < a.n_mats; ++i) {
        a.tile0[i] = cols / 16u;
        cols += a.mats[i].cols;
        if (a.mats[i].cols % 64u) return set_error(XP_E_ARG, "%s: cols=%u", who, a.mats[i].cols);
    }
    if (geglu) cols = a.mats[0].cols;
    if (a.nblk % 4u || cols % bn || p.n_tiles * bn != cols || (fmt != XP_SCALE_F16_QUAD && fmt != XP_SCALE_BF16_QUAD))
        return set_error(XP_E_ARG, "%s: shape outside the prefill GEMM's", who);
    if (fmt == XP_SCALE_F16_QUAD) gemm_launch<XP_SCALE_F16_QUAD>(a, p.shape, geglu, st);
    else gemm_launch<XP_SCALE_BF16_QUAD>(a, p.shape, geglu, st);
    return launched(who);
}

int launch_pf_qk(const PfQkArgs& a, float theta, hipStream_t st) {
    RopeFreq f;
    rope_freq(f, 256, theta);
    const uint32_t waves = a.rows * (a.n_heads + 2u * a.kv_heads);
    hipLaunchKernelGGL(pf_qk_kernel, dim3((waves + 3u) / 4u), dim3(256), 0, st, a, f);
    return launched("prefill qk");
}

// Key splits of an attention launch: enough workgroups for the CUs when the
// rows alone give few, each split at least two 128-key tiles long.
uint32_t pf_attn_splits(uint32_t rows, uint32_t group, uint32_t kv_heads, uint32_t max_keys, int n_cu) {
    const uint32_t wgs = (rows * group + 31u) / 32u * kv_heads, tiles = (max_keys + kPaKeys - 1u) / kPaKeys;
    const uint32_t want = uint32_t(n_cu > 0 ? n_cu : 256) / std::max(wgs, 1u);
    return std::max(1u, std::min(want, tiles / 2u));
}

int launch_pf_attn(const PfAttnArgs& a, uint32_t group, uint32_t splits, hipStream_t st) {
    const dim3 g1((a.rows * group + 31u) / 32u, a.kv_heads, 1), g(g1.x, g1.y, splits);
#define XP_PA(G)                                                                                        \
    do {                                                                                                \
        hipLaunchKernelGGL((pf_attn_kernel<G>), g, dim3(kPaThreads), 0, st, a);                                \
        if (splits > 1u) hipLaunchKernelGGL((pf_attn_combine_kernel<G>), g1, dim3(256), 0, st, a, splits); \
    } while (0)
    if (group == 1u) XP_PA(1);
    else if (group == 2u) XP_PA(2);
    else if (group == 4u) XP_PA(4);
    else return set_error(XP_E_ARG, "prefill attention: %u query heads per kv head (1, 2 or 4)", group);
#undef XP_PA
    return launched("prefill attention");
}

}  // namespace xp
