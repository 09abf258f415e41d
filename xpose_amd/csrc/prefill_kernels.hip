// Prefill-shaped twins of the decode kernels (kernels/llm_sampling.cl:496-736):
// row-indexed softmax, causal / sliding-window attention scores and apply,
// row RMSNorm, per-head row QK-norm, per-row-position RoPE, KV row append and
// embedding row gather, each behind its own C-ABI entry.
//
// The reference gives row reductions one thread per row (serial loops over
// the columns); here a row is one wave: lanes stride over the columns and DPP
// wave reductions combine them. Scores and apply are fp32 products on the
// matrix cores (v_mfma_f32_32x32x2_f32), the rest elementwise.
// Layouts are the reference's, row-major: row r occupies [r n_cols, (r + 1)
// n_cols); q, scores and outputs are [head][query][...]; caches [t][kv_head][d]
// in fp32.
#include <algorithm>
#include <cmath>

#include "xp_device.hpp"
#include "xp_launch.hpp"

namespace xp {
namespace {

constexpr int kPfThreads = 256;
constexpr int kPfWaves = kPfThreads / kWave;

uint32_t pf_blocks(size_t n) {
    return uint32_t(std::min<size_t>((n + kPfThreads - 1) / kPfThreads, 65536));
}
uint32_t pf_row_blocks(size_t rows) { return uint32_t((rows + kPfWaves - 1) / kPfWaves); }

// softmax_rows_stats (llm_sampling.cl:527-547): one wave per row, up to 2048
// columns held in registers between the maximum and the sum, so that a row
// is read once (4096 x 2024: 24 -> 9.9 us). A row takes the time of its
// registers, filled or not, so it gets the next power of two of 64 columns (a
// row of 65 to 500 in 32 registers: 4000 rows 6.0 us, in its own 3.7).
template <int kSmRegs>
__global__ __launch_bounds__(kPfThreads) void softmax_rows_stats_kernel(float* stats, const float* x,
                                                                       uint32_t n_rows, uint32_t n_cols) {
    const uint32_t r = blockIdx.x * kPfWaves + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (r >= n_rows) return;   // whole waves
    const float* row = x + size_t(r) * n_cols;
    const bool held = n_cols <= uint32_t(kSmRegs * kWave);
    float v[kSmRegs];
    float m = -INFINITY;
    if (held) {
#pragma unroll
        for (int j = 0; j < kSmRegs; ++j) {
            const uint32_t c = lane + uint32_t(j) * kWave;
            v[j] = c < n_cols ? row[c] : -INFINITY;
        }
#pragma unroll
        for (int j = 0; j < kSmRegs; ++j) m = fmaxf(m, v[j]);
    } else {
        for (uint32_t j = lane; j < n_cols; j += kWave) m = fmaxf(m, row[j]);
    }
    m = wave_max(m);
    if (!isfinite(m)) {
        if (lane == 0) {
            stats[2 * size_t(r)] = 0.0f;
            stats[2 * size_t(r) + 1] = 1.0f;
        }
        return;
    }
    float s = 0.0f;
    if (held) {
#pragma unroll
        for (int j = 0; j < kSmRegs; ++j)
            if (uint32_t(j) * kWave < n_cols) s += expf(v[j] - m);   // columns past the end add 0
    } else {
        for (uint32_t j = lane; j < n_cols; j += kWave) s += expf(row[j] - m);
    }
    s = wave_sum(s);
    if (lane == 0) {
        stats[2 * size_t(r)] = m;
        stats[2 * size_t(r) + 1] = s;
    }
}

// softmax_rows_apply (llm_sampling.cl:549-556): a wave takes a run of
// kSmRun columns of one row (no division per element to find the row; eight
// loads in flight a lane). Where runs are mostly past the row's end, or too few
// for the CUs, a thread takes one element. Runs / elements in us: 16000 rows of
// 65 5.2 / 3.6, of 129 6.5 / 5.4, of 200 7.1 / 7.6; 1000 rows of 1000 4.2 / 3.6,
// of 2024 5.1 / 5.3; 4000 rows of 2024 12.2 / 16.0.
constexpr size_t kSmFew = 3u << 19;   // elements
__global__ void softmax_elems_apply_kernel(float* x, const float* stats, uint32_t n_cols, size_t total) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += size_t(gridDim.x) * blockDim.x) {
        const size_t r = i / n_cols;
        x[i] = expf(x[i] - stats[2 * r]) / stats[2 * r + 1];
    }
}
constexpr uint32_t kSmRun = 8 * kWave;
__global__ __launch_bounds__(kPfThreads) void softmax_rows_apply_kernel(float* x, const float* stats, uint32_t n_cols,
                                                                       uint32_t runs, size_t n_runs) {
    const uint32_t lane = threadIdx.x % kWave;
    for (size_t i = size_t(blockIdx.x) * kPfWaves + threadIdx.x / kWave; i < n_runs;
         i += size_t(gridDim.x) * kPfWaves) {
        const size_t r = i / runs;
        const uint32_t c0 = uint32_t(i - r * runs) * kSmRun + lane;
        const float m = stats[2 * r], s = stats[2 * r + 1];
        float* row = x + r * n_cols;
        float v[kSmRun / kWave];
#pragma unroll
        for (uint32_t j = 0; j < kSmRun / kWave; ++j) v[j] = c0 + j * kWave < n_cols ? row[c0 + j * kWave] : 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < kSmRun / kWave; ++j)
            if (c0 + j * kWave < n_cols) row[c0 + j * kWave] = expf(v[j] - m) / s;
    }
}

// ---- attention products -----------------------------------------------------
// fp32 operands on v_mfma_f32_32x32x2_f32: fp32 products and sums throughout,
// at the card's fp32 rate (154 TFLOP/s measured on a large product), where one
// thread an element, with nothing reused, made 550 us of 2.1 GFLOP of scores
// and 774 us of the apply. The query heads of one kv head are consecutive
// rows of q, scores and out, so a tile's rows are rows of that whole group.
//
// Operand lanes: row (A) or column (B) lane % 32, and of the eight k a step of
// four instructions takes, 4 (lane / 32) + 0..3, one 16-byte LDS read. C: column
// lane % 32, rows 8 i + 4 (lane / 32) + r in word 4 i + r.
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr uint32_t kAsRows = 32, kAsKeys = 64, kAsDims = 64, kAsStride = kAsDims + 4;   // floats; rows 4 banks apart
constexpr uint32_t kAsOut = kAsKeys + 4;
struct __attribute__((aligned(16))) AsSmem {
    union {
        struct {
            float q[kAsRows * kAsStride], k[kAsKeys * kAsStride];
        } t;
        float o[2][kAsRows * kAsOut];                     // the two halves of the dims
    };
};

// attention_scores_prefill (llm_sampling.cl:574-600): causal and window masks
// folded in. A workgroup makes 32 x 64 scores, 64 dims of both sides in LDS at
// a time, the next on their way; a wave 32 x 32 of them over half of the dims
// there. Small tiles: one is a chain of loads, barriers and 64-cycle
// instructions that only other workgroups fill, so four share a CU. The halves
// meet in LDS, from where a wave writes whole rows, the masks scalar but for
// the key. A tile that the masks leave nothing of is only filled, by a workgroup
// that has other key tiles of the row to make. From 8 row tiles on the grid's x
// is a multiple of 8, so the tiles of one row, whose runs share cache lines, are
// written through one XCD's L2. 1024 queries over 2024 keys, window 512, 4 heads: 24 us,
// where 64 x 64 tiles took 38, a workgroup for each 32 x 64 tile 35 and one
// thread a score 550 (the matrix units work 8, the 33 MB out take 7).
__global__ __launch_bounds__(kPfThreads, 4) void attention_scores_prefill_kernel(
    float* scores, const float* q, const float* kc, uint32_t group, uint32_t kv_heads, uint32_t head_dim,
    uint32_t n_query, uint32_t seq_len, uint32_t q_offset, uint32_t window, float scale) {
    __shared__ AsSmem sm;
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const uint32_t c32 = lane % 32u, half = lane / 32u;
    const size_t rows = size_t(group) * n_query;          // of this kv head
    for (uint64_t tb = uint64_t(blockIdx.y) * kAsKeys; tb < seq_len; tb += uint64_t(gridDim.y) * kAsKeys)
    for (uint32_t kvh = blockIdx.z; kvh < kv_heads; kvh += gridDim.z)
    for (size_t r0 = size_t(blockIdx.x) * kAsRows; r0 < rows; r0 += size_t(gridDim.x) * kAsRows) {
        const uint32_t t0 = uint32_t(tb);
        // the positions of the tile's queries: one run, or two where it
        // crosses from one head to the next (then any position)
        const uint32_t nr = uint32_t(rows - r0 < kAsRows ? rows - r0 : kAsRows);
        const uint32_t nk = min(seq_len - t0, kAsKeys);
        const uint32_t qa = uint32_t(r0 % n_query);
        const bool one = uint64_t(qa) + nr <= n_query;
        const uint64_t plo = uint64_t(q_offset) + (one ? qa : 0u), phi = uint64_t(q_offset) + (one ? qa + nr : n_query) - 1u;
        // (positions wrap at 2^32, as the reference's; a tile that could is not left out)
        const bool dead = phi <= 0xFFFFFFFFull && (t0 > phi || (window != 0u && uint64_t(t0) + nk - 1u + window <= plo));
        const uint32_t t = t0 + lane;
        float* ob = scores + (size_t(kvh) * rows + r0) * seq_len + t;
        if (dead) {
            for (uint32_t r = wave; r < nr; r += kPfWaves)
                if (lane < nk) ob[size_t(r) * seq_len] = -INFINITY;
            continue;
        }
        // word i of a chunk: row i / 16, dims 4 (i % 16) ..; rows past the end
        // repeat the last one, their scores are not stored; dims past the end
        // are zeros
        constexpr uint32_t W = kAsDims / 4u, RS = kPfThreads / W, UQ = kAsRows / RS, UK = kAsKeys / RS;
        const uint32_t lr = tid / W, ld = (tid % W) * 4u;
        const float* qp[UQ];
        const float* kp[UK];
#pragma unroll
        for (uint32_t j = 0; j < UQ; ++j) qp[j] = q + (size_t(kvh) * rows + r0 + min(lr + j * RS, nr - 1u)) * head_dim;
#pragma unroll
        for (uint32_t j = 0; j < UK; ++j) kp[j] = kc + (size_t(t0 + min(lr + j * RS, nk - 1u)) * kv_heads + kvh) * head_dim;
        u32x4 qr[UQ], kr[UK];
        auto load = [&](uint32_t d0) {
            const uint32_t d = min(d0 + ld, head_dim - 4u);
#pragma unroll
            for (uint32_t j = 0; j < UQ; ++j) qr[j] = *reinterpret_cast<const u32x4*>(qp[j] + d);
#pragma unroll
            for (uint32_t j = 0; j < UK; ++j) kr[j] = *reinterpret_cast<const u32x4*>(kp[j] + d);
        };
        // two sums a wave, with the waves' halves four of head_dim / 4 dims:
        // shorter chains round less
        f32x16 acc[2];
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][i] = 0.0f;
        load(0);
        for (uint32_t d0 = 0; d0 < head_dim; d0 += kAsDims) {
            const u32x4 zero{0u, 0u, 0u, 0u};
            const bool in = d0 + ld < head_dim;
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < UQ; ++j) *reinterpret_cast<u32x4*>(sm.t.q + (lr + j * RS) * kAsStride + ld) = in ? qr[j] : zero;
#pragma unroll
            for (uint32_t j = 0; j < UK; ++j) *reinterpret_cast<u32x4*>(sm.t.k + (lr + j * RS) * kAsStride + ld) = in ? kr[j] : zero;
            __syncthreads();
            if (d0 + kAsDims < head_dim) load(d0 + kAsDims);
            const uint32_t dw = (wave / 2u) * (kAsDims / 2u) + 4u * half;
            const float* A = sm.t.q + c32 * kAsStride + dw;
            const float* B = sm.t.k + (wave % 2u * 32u + c32) * kAsStride + dw;
#pragma unroll
            for (uint32_t d = 0; d < kAsDims / 2u; d += 8) {
                const float4 x = *reinterpret_cast<const float4*>(A + d), y = *reinterpret_cast<const float4*>(B + d);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, acc[1], 0, 0, 0);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, acc[1], 0, 0, 0);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t r = 8u * uint32_t(i / 4) + 4u * half + uint32_t(i % 4);
            sm.o[wave / 2u][r * kAsOut + wave % 2u * 32u + c32] = acc[0][i] + acc[1][i];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t i = 0; i < kAsRows / kPfWaves; ++i) {
            const uint32_t r = wave + kPfWaves * i;
            const float s = (sm.o[0][r * kAsOut + lane] + sm.o[1][r * kAsOut + lane]) * scale;
            const uint32_t qi = one ? qa + r : (qa + r) % n_query, qpos = q_offset + qi;
            const bool off = t > qpos || (window != 0u && t + window <= qpos);
            if (r < nr && lane < nk) ob[size_t(r) * seq_len] = off ? -INFINITY : s;
        }
        __syncthreads();
    }
}

// attention_apply_prefill (llm_sampling.cl:605-627). A workgroup makes 32 rows x
// 32 NT dims, its eight waves 32 keys of each 256: a wave's probabilities pass
// through LDS of its own (no barrier), a lane reads NT dims of a key's row
// at once (dims NT c + n are column c of tile n), and the waves' sums are added
// at the end in wave order. Latency bounds it: the next 32 keys are on their
// way. Where a wave's 32 x 32 probabilities are all zero (masked keys: most of
// a causal or windowed prompt) and its 32 rows of v are finite, the products
// are zeros and are left out. 1024 queries over 2024 keys,
// window 512, 4 heads: 774 -> 26 us.
constexpr uint32_t kApThreads = 512, kApWaves = kApThreads / kWave;
constexpr uint32_t kApKeys = 32, kApRows = 32, kApPs = kApKeys + 4;
template <uint32_t NT>
struct __attribute__((aligned(16))) ApSmem {
    union {
        float p[kApWaves][kApRows * kApPs];
        float o[kApWaves][kApRows][32 * NT];
    };
};
template <uint32_t NT>
__global__ __launch_bounds__(kApThreads, 8 / NT) void attention_apply_prefill_kernel(
    float* out, const float* probs, const float* vc, uint32_t group, uint32_t kv_heads, uint32_t head_dim,
    uint32_t n_query, uint32_t seq_len) {
    typedef uint32_t vec __attribute__((ext_vector_type(NT)));
    constexpr uint32_t kApDims = 32 * NT;
    __shared__ ApSmem<NT> sm;
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const uint32_t c32 = lane % 32u, half = lane / 32u;
    const size_t rows = size_t(group) * n_query;
    const uint32_t d = blockIdx.y * kApDims + NT * c32;
    const bool dlive = d < head_dim;                      // whole lanes: head_dim is a multiple of 4
    const uint32_t vst = kv_heads * head_dim;
    for (uint32_t kvh = blockIdx.z; kvh < kv_heads; kvh += gridDim.z)
    for (size_t r0 = size_t(blockIdx.x) * kApRows; r0 < rows; r0 += size_t(gridDim.x) * kApRows) {
        const uint32_t nr = uint32_t(rows - r0 < kApRows ? rows - r0 : kApRows);
        // raw buffers, a descriptor a row of loads (scalar arithmetic only):
        // what lies past the rows or the dims reads as zero (offsets below
        // 2^32, which the caller checks)
        auto from = [](const float* base, uint32_t off, uint32_t end) {
            off = __builtin_amdgcn_readfirstlane(min(off, end));
            return make_rsrc(reinterpret_cast<const unsigned char*>(base) + off, __builtin_amdgcn_readfirstlane(end - off));
        };
        const float* pb = probs + (size_t(kvh) * rows + r0) * seq_len;
        const float* vb = vc + size_t(kvh) * head_dim;
        const uint32_t pend = nr * seq_len * 4u, vend = (seq_len * vst - kvh * head_dim) * 4u;
        const uint32_t vo = dlive ? (4u * half * vst + d) * 4u : 0xF0000000u;
        f32x16 acc[NT];
#pragma unroll
        for (uint32_t n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][i] = 0.0f;
        float* ps = sm.p[wave];
        uint32_t pr[16];                                  // row 2 j + half, key c32 of the chunk
        auto load_p = [&](uint32_t t0) {
            const uint32_t t = t0 + c32, o = t < seq_len ? (half * seq_len + t) * 4u : 0xF0000000u;
#pragma unroll
            for (uint32_t j = 0; j < 16; ++j) pr[j] = __builtin_amdgcn_raw_buffer_load_b32(from(pb, 8u * j * seq_len, pend), int(o), 0, 0);
        };
        // instruction (s, j) of a chunk takes keys 8 s + j and 8 s + 4 + j
        auto load_v = [&](uint32_t t0, uint32_t i) {
            const rsrc_t rv = from(vb, (t0 + 8u * (i / 4u) + i % 4u) * vst * 4u, vend);
            if constexpr (NT == 4) return __builtin_amdgcn_raw_buffer_load_b128(rv, int(vo), 0, 0);
            else return __builtin_amdgcn_raw_buffer_load_b64(rv, int(vo), 0, 0);
        };
        constexpr uint32_t kStep = kApWaves * kApKeys;
        vec v[16];
        uint32_t t0 = wave * kApKeys;
        if (t0 < seq_len) {
            load_p(t0);
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) v[i] = load_v(t0, i);
        }
        for (; t0 < seq_len; t0 += kStep) {
            uint32_t any = 0;
#pragma unroll
            for (uint32_t j = 0; j < 16; ++j) {
                any |= pr[j] << 1;                        // not the sign: -0 is zero
                ps[(2u * j + half) * kApPs + c32] = __uint_as_float(pr[j]);
            }
            load_p(t0 + kStep);
            bool work = __ballot(any != 0u) != 0ull;
            if (!work) {
                uint32_t big = 0;
#pragma unroll
                for (uint32_t i = 0; i < 16; ++i)
#pragma unroll
                    for (uint32_t n = 0; n < NT; ++n) big = max(big, v[i][n] << 1);
                work = __ballot(big >= 0xFF000000u) != 0ull;   // an infinity or NaN: 0 v is not 0
            }
            if (work) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (uint32_t st = 0; st < 4; ++st) {
                    const float4 x = *reinterpret_cast<const float4*>(ps + c32 * kApPs + 8u * st + 4u * half);
                    const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
                        for (uint32_t n = 0; n < NT; ++n)
                            acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[j], __uint_as_float(v[4u * st + j][n]), acc[n], 0, 0, 0);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) v[i] = load_v(t0 + kStep, i);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t r = 8u * uint32_t(i / 4) + 4u * half + uint32_t(i % 4);
            vec x;
#pragma unroll
            for (uint32_t n = 0; n < NT; ++n) x[n] = __float_as_uint(acc[n][i]);
            *reinterpret_cast<vec*>(&sm.o[wave][r][NT * c32]) = x;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t i = tid; i < kApRows * kApDims / 4u; i += kApThreads) {
            const uint32_t r = i / (kApDims / 4u), c = i % (kApDims / 4u), dd = blockIdx.y * kApDims + 4u * c;
            float4 s = *reinterpret_cast<const float4*>(&sm.o[0][r][4u * c]);
#pragma unroll
            for (uint32_t w = 1; w < kApWaves; ++w) {
                const float4 e = *reinterpret_cast<const float4*>(&sm.o[w][r][4u * c]);
                s.x += e.x; s.y += e.y; s.z += e.z; s.w += e.w;
            }
            if (r < nr && dd < head_dim)
                *reinterpret_cast<float4*>(out + (size_t(kvh) * rows + r0 + r) * head_dim + dd) = s;
        }
        __syncthreads();
    }
}
// The same with one thread per output element, for a head_dim that is not a
// multiple of 4, values or an output that are not 16-byte aligned, or values
// or probability rows whose byte offsets pass 2^32.
__global__ void attention_apply_prefill_scalar_kernel(float* out, const float* probs, const float* vc,
                                                      uint32_t n_heads, uint32_t kv_heads, uint32_t head_dim,
                                                      uint32_t n_query, uint32_t seq_len, size_t total) {
    const uint32_t group = n_heads / kv_heads, vstride = kv_heads * head_dim;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += size_t(gridDim.x) * blockDim.x) {
        const uint32_t d = uint32_t(i % head_dim);
        const size_t hq = i / head_dim;
        const uint32_t qi = uint32_t(hq % n_query), h = uint32_t(hq / n_query);
        const float* p = probs + (size_t(h) * n_query + qi) * seq_len;
        const float* v = vc + size_t(h / group) * head_dim + d;
        float a0 = 0.0f, a1 = 0.0f;
        uint32_t t = 0;
        for (; t + 2 <= seq_len; t += 2) {
            a0 = fmaf(p[t], v[size_t(t) * vstride], a0);
            a1 = fmaf(p[t + 1], v[size_t(t + 1) * vstride], a1);
        }
        if (t < seq_len) a0 = fmaf(p[t], v[size_t(t) * vstride], a0);
        out[i] = a0 + a1;
    }
}

// rmsnorm_rows_sumsq (llm_sampling.cl:634-642): one wave per row.
__global__ __launch_bounds__(kPfThreads) void rmsnorm_rows_sumsq_kernel(float* rowss, const float* in,
                                                                       uint32_t n_rows, uint32_t n) {
    const uint32_t r = blockIdx.x * kPfWaves + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (r >= n_rows) return;
    const float* row = in + size_t(r) * n;
    float ss = 0.0f;
    for (uint32_t j = lane; j < n; j += kWave) ss = fmaf(row[j], row[j], ss);
    ss = wave_sum(ss);
    if (lane == 0) rowss[r] = ss;
}

// rmsnorm_rows_apply_gemma (llm_sampling.cl:645-656).
__global__ void rmsnorm_rows_apply_gemma_kernel(float* out, const float* in, const float* w,
                                                const float* rowss, uint32_t n, float eps, size_t total) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += size_t(gridDim.x) * blockDim.x) {
        const size_t r = i / n;
        const float scale = rsq_hw(rowss[r] / float(n) + eps);
        out[i] = in[i] * scale * (1.0f + w[i - r * n]);
    }
}

// rmsnorm_heads_rows_gemma (llm_sampling.cl:659-672): one wave per
// (token, head) row of head_dim.
__global__ __launch_bounds__(kPfThreads) void rmsnorm_heads_rows_gemma_kernel(
    float* out, const float* in, const float* w, uint32_t n_rows, uint32_t head_dim, float eps) {
    const uint32_t r = blockIdx.x * kPfWaves + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (r >= n_rows) return;
    const float* row = in + size_t(r) * head_dim;
    float ss = 0.0f;
    for (uint32_t j = lane; j < head_dim; j += kWave) ss = fmaf(row[j], row[j], ss);
    const float scale = rsq_hw(wave_sum(ss) / float(head_dim) + eps);
    for (uint32_t j = lane; j < head_dim; j += kWave) out[size_t(r) * head_dim + j] = row[j] * scale * (1.0f + w[j]);
}

// rope_prefill (llm_sampling.cl:687-708): one thread per rotated pair, token
// ti at position pos0 + ti, with the decode rope's inverse frequencies, so a
// row rotates exactly as xp_rope rotates it at that position.
__global__ void rope_prefill_kernel(float* x, uint32_t n_heads, uint32_t head_dim, uint32_t pos0,
                                    RopeFreq f, size_t total) {
    const uint32_t hdhalf = head_dim / 2u;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += size_t(gridDim.x) * blockDim.x) {
        const uint32_t d = uint32_t(i % hdhalf);
        const size_t th = i / hdhalf;
        const uint32_t ti = uint32_t(th / n_heads);
        const size_t base = th * head_dim + d;
        const float ang = float(pos0 + ti) * f.inv[d];
        float s, c;
        sincosf(ang, &s, &c);
        const float a = x[base], b = x[base + hdhalf];
        x[base] = a * c - b * s;
        x[base + hdhalf] = b * c + a * s;
    }
}

// kv_append_rows (llm_sampling.cl:714-721).
__global__ void kv_append_rows_kernel(float* dst, const float* src, size_t total) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += size_t(gridDim.x) * blockDim.x)
        dst[i] = src[i];
}

// embed_lookup_rows (llm_sampling.cl:728-736); an id past the table writes
// zeros instead of reading past it.
__global__ void embed_lookup_rows_kernel(float* out, const float* table, const uint32_t* tokens,
                                         uint32_t n, uint32_t vocab, size_t total) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += size_t(gridDim.x) * blockDim.x) {
        const size_t ti = i / n;
        const uint32_t tok = tokens[ti];
        out[i] = tok < vocab ? table[size_t(tok) * n + (i - ti * n)] : 0.0f;
    }
}

int launched(const char* who) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(XP_E_HIP, "%s: launch -> %s", who, hipGetErrorString(e));
    return XP_OK;
}

}  // namespace
}  // namespace xp

using namespace xp;

extern "C" {

int xp_softmax_rows_stats(float* stats, const float* x, uint32_t n_rows, uint32_t n_cols,
                          xp_stream stream) {
    XP_REQUIRE(stats && x, "null pointer");
    XP_REQUIRE(n_rows > 0 && n_cols > 0, "empty shape %u x %u", n_rows, n_cols);
    const uint32_t regs = (n_cols - 1u) / kWave + 1u;   // a lane's columns
#define XP_SM(R)                                                                                                        \
    hipLaunchKernelGGL(softmax_rows_stats_kernel<R>, dim3(pf_row_blocks(n_rows)), dim3(kPfThreads), 0, as_stream(stream), \
                       stats, x, n_rows, n_cols)
    if (regs <= 1u) XP_SM(1);
    else if (regs <= 2u) XP_SM(2);
    else if (regs <= 4u) XP_SM(4);
    else if (regs <= 8u) XP_SM(8);
    else if (regs <= 16u) XP_SM(16);
    else XP_SM(32);
#undef XP_SM
    return launched("xp_softmax_rows_stats");
}

int xp_softmax_rows_apply(float* x, const float* stats, uint32_t n_rows, uint32_t n_cols,
                          xp_stream stream) {
    XP_REQUIRE(stats && x, "null pointer");
    XP_REQUIRE(n_rows > 0 && n_cols > 0, "empty shape %u x %u", n_rows, n_cols);
    const size_t total = size_t(n_rows) * n_cols;
    if (n_cols < 192u || total <= kSmFew) {
        hipLaunchKernelGGL(softmax_elems_apply_kernel, dim3(pf_blocks(total)), dim3(kPfThreads), 0, as_stream(stream), x,
                           stats, n_cols, total);
        return launched("xp_softmax_rows_apply");
    }
    const uint32_t runs = (n_cols - 1u) / kSmRun + 1u;
    const size_t n_runs = size_t(n_rows) * runs;
    hipLaunchKernelGGL(softmax_rows_apply_kernel, dim3(uint32_t(std::min<size_t>((n_runs + kPfWaves - 1) / kPfWaves, 65536))),
                       dim3(kPfThreads), 0, as_stream(stream), x, stats, n_cols, runs, n_runs);
    return launched("xp_softmax_rows_apply");
}

int xp_attention_scores_prefill(float* scores, const float* q, const float* kcache, uint32_t n_heads,
                                uint32_t kv_heads, uint32_t head_dim, uint32_t n_query,
                                uint32_t seq_len, uint32_t q_offset, uint32_t window, float scale,
                                xp_stream stream) {
    XP_REQUIRE(scores && q && kcache, "null pointer");
    XP_REQUIRE(n_heads > 0 && kv_heads > 0 && n_heads % kv_heads == 0,
               "n_heads=%u must be a positive multiple of kv_heads=%u", n_heads, kv_heads);
    XP_REQUIRE(head_dim > 0 && head_dim % 4 == 0, "head_dim=%u must be a positive multiple of 4", head_dim);
    XP_REQUIRE(n_query > 0 && seq_len > 0, "n_query=%u, seq_len=%u must be positive", n_query, seq_len);
    XP_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kcache)) & 15u) == 0,
               "q and kcache must be 16-byte aligned");
    const uint32_t group = n_heads / kv_heads;
    const size_t qt = (size_t(group) * n_query - 1u) / kAsRows + 1u;
    // fewer than 8 row tiles are not rounded up: workgroups without one would
    // take places that the key tiles need (8 kv heads of 64, one query over 8000
    // keys: 34 us so, 6.4 without)
    const uint32_t gx = uint32_t(qt < 8u ? qt : std::min<size_t>((qt + 7u) / 8u * 8u, 1u << 20)), gz = std::min(kv_heads, 65535u);
    // key tiles of a row spread over as many workgroups as the CUs hold at
    // once (four each): the filled ones then cost no launch of their own
    const uint32_t gy = uint32_t(std::min<uint64_t>(std::min((seq_len - 1u) / kAsKeys + 1u, 65535u),
                                                    1024u / std::min<uint64_t>(uint64_t(gx) * gz, 1024u)));
    hipLaunchKernelGGL(attention_scores_prefill_kernel, dim3(gx, gy, gz), dim3(kPfThreads), 0, as_stream(stream), scores,
                       q, kcache, group, kv_heads, head_dim, n_query, seq_len, q_offset, window, scale);
    return launched("xp_attention_scores_prefill");
}

int xp_attention_apply_prefill(float* out, const float* probs, const float* vcache, uint32_t n_heads,
                               uint32_t kv_heads, uint32_t head_dim, uint32_t n_query,
                               uint32_t seq_len, xp_stream stream) {
    XP_REQUIRE(out && probs && vcache, "null pointer");
    XP_REQUIRE(n_heads > 0 && kv_heads > 0 && n_heads % kv_heads == 0,
               "n_heads=%u must be a positive multiple of kv_heads=%u", n_heads, kv_heads);
    XP_REQUIRE(head_dim > 0 && n_query > 0 && seq_len > 0, "empty shape");
    const uint32_t group = n_heads / kv_heads;
    // the tiled kernel's offsets run up to 288 keys past the end, with room for
    // the one that marks a lane past the dims
    const uint64_t vbytes = (uint64_t(seq_len) + 512u) * kv_heads * head_dim * 4u, pbytes = (uint64_t(seq_len) + 512u) * 33u * 4u;
    const bool tiled = head_dim % 4u == 0 && (head_dim - 1u) / 64u + 1u <= 65535u && vbytes < 0xE0000000ull &&
                       pbytes < 0xE0000000ull && ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(vcache)) & 15u) == 0;
    if (tiled) {
        const size_t rt = (size_t(group) * n_query - 1u) / kApRows + 1u;
        const uint32_t gx = uint32_t(std::min<size_t>((rt + 7u) / 8u * 8u, 1u << 20)), gz = std::min(kv_heads, 65535u);
        // 128 dims a workgroup read p half as often; where that gives the 256
        // CUs less than one each, 64 dims are the shorter chain (26 against 31 us
        // at 1024 queries over 2024 keys, 8.5 against 6.3 at 200)
        const uint32_t wide = (head_dim - 1u) / 128u + 1u;
        if (rt * wide * kv_heads >= 256u)
            hipLaunchKernelGGL(attention_apply_prefill_kernel<4>, dim3(gx, wide, gz), dim3(kApThreads), 0, as_stream(stream),
                               out, probs, vcache, group, kv_heads, head_dim, n_query, seq_len);
        else
            hipLaunchKernelGGL(attention_apply_prefill_kernel<2>, dim3(gx, (head_dim - 1u) / 64u + 1u, gz), dim3(kApThreads),
                               0, as_stream(stream), out, probs, vcache, group, kv_heads, head_dim, n_query, seq_len);
    } else {
        const size_t total = size_t(n_heads) * n_query * head_dim;
        hipLaunchKernelGGL(attention_apply_prefill_scalar_kernel, dim3(pf_blocks(total)), dim3(kPfThreads), 0,
                           as_stream(stream), out, probs, vcache, n_heads, kv_heads, head_dim, n_query, seq_len, total);
    }
    return launched("xp_attention_apply_prefill");
}

int xp_rmsnorm_rows_sumsq(float* rowss, const float* in, uint32_t n_rows, uint32_t n,
                          xp_stream stream) {
    XP_REQUIRE(rowss && in, "null pointer");
    XP_REQUIRE(n_rows > 0 && n > 0, "empty shape %u x %u", n_rows, n);
    hipLaunchKernelGGL(rmsnorm_rows_sumsq_kernel, dim3(pf_row_blocks(n_rows)), dim3(kPfThreads), 0,
                       as_stream(stream), rowss, in, n_rows, n);
    return launched("xp_rmsnorm_rows_sumsq");
}

int xp_rmsnorm_rows_apply_gemma(float* out, const float* in, const float* w, const float* rowss,
                                uint32_t n_rows, uint32_t n, float eps, xp_stream stream) {
    XP_REQUIRE(out && in && w && rowss, "null pointer");
    XP_REQUIRE(n_rows > 0 && n > 0, "empty shape %u x %u", n_rows, n);
    const size_t total = size_t(n_rows) * n;
    hipLaunchKernelGGL(rmsnorm_rows_apply_gemma_kernel, dim3(pf_blocks(total)), dim3(kPfThreads), 0,
                       as_stream(stream), out, in, w, rowss, n, eps, total);
    return launched("xp_rmsnorm_rows_apply_gemma");
}

int xp_rmsnorm_heads_rows_gemma(float* out, const float* in, const float* w, uint32_t n_tokens,
                                uint32_t n_heads, uint32_t head_dim, float eps, xp_stream stream) {
    XP_REQUIRE(out && in && w, "null pointer");
    XP_REQUIRE(n_tokens > 0 && n_heads > 0 && head_dim > 0, "empty shape");
    XP_REQUIRE(out != in, "out must not alias in (each row is read after other lanes write)");
    const size_t rows = size_t(n_tokens) * n_heads;
    XP_REQUIRE(rows <= 0xFFFFFFFFull, "too many rows");
    hipLaunchKernelGGL(rmsnorm_heads_rows_gemma_kernel, dim3(pf_row_blocks(rows)), dim3(kPfThreads), 0,
                       as_stream(stream), out, in, w, uint32_t(rows), head_dim, eps);
    return launched("xp_rmsnorm_heads_rows_gemma");
}

int xp_rope_prefill(float* x, uint32_t n_tokens, uint32_t n_heads, uint32_t head_dim, uint32_t pos0,
                    float theta, xp_stream stream) {
    XP_REQUIRE(x, "null pointer");
    XP_REQUIRE(n_tokens > 0 && n_heads > 0 && head_dim > 0 && head_dim % 2 == 0 &&
                   head_dim <= uint32_t(kMaxHeadDim),
               "empty shape, or head_dim=%u odd or above %d", head_dim, kMaxHeadDim);
    XP_REQUIRE(theta > 0.0f, "theta=%g must be positive", double(theta));
    RopeFreq f;
    rope_freq(f, head_dim, theta);
    const size_t total = size_t(n_tokens) * n_heads * (head_dim / 2);
    hipLaunchKernelGGL(rope_prefill_kernel, dim3(pf_blocks(total)), dim3(kPfThreads), 0,
                       as_stream(stream), x, n_heads, head_dim, pos0, f, total);
    return launched("xp_rope_prefill");
}

int xp_kv_append_rows(float* cache, const float* src, uint32_t n_tokens, uint32_t row, uint32_t pos0,
                      xp_stream stream) {
    XP_REQUIRE(cache && src, "null pointer");
    XP_REQUIRE(n_tokens > 0 && row > 0, "empty shape");
    const size_t total = size_t(n_tokens) * row;
    hipLaunchKernelGGL(kv_append_rows_kernel, dim3(pf_blocks(total)), dim3(kPfThreads), 0,
                       as_stream(stream), cache + size_t(pos0) * row, src, total);
    return launched("xp_kv_append_rows");
}

int xp_embed_lookup_rows(float* out, const float* table, const uint32_t* tokens, uint32_t n_tokens,
                         uint32_t n, uint32_t vocab, xp_stream stream) {
    XP_REQUIRE(out && table && tokens, "null pointer");
    XP_REQUIRE(n_tokens > 0 && n > 0 && vocab > 0, "empty shape");
    const size_t total = size_t(n_tokens) * n;
    hipLaunchKernelGGL(embed_lookup_rows_kernel, dim3(pf_blocks(total)), dim3(kPfThreads), 0,
                       as_stream(stream), out, table, tokens, n, vocab, total);
    return launched("xp_embed_lookup_rows");
}

}  // extern "C"
