// The full-vocabulary sampling chain (kernels/llm_sampling.cl:130-225,
// 257-281, 349-386, 399-488): temperature, the strided-chain max / exp-sum
// softmax, per-chain top-k with rank selection, the top-k mask, top-p and the
// two multinomial draws. In the reference these are verified building blocks
// that decode does not call; here each is one gfx950 kernel behind an
// xp_<name> entry point with the reference's argument meaning.
//
// Every kernel evaluates what the reference evaluates in the same order where
// the order shows: a chain's sum is added in chain order, the serial
// finalisers stay serial. Sums, comparisons, the division and the cumulative
// walks are therefore bit-identical to the reference's fp32 arithmetic on the
// same inputs; only exp (the device libm against llvmpipe's) can differ in the
// last bits. What has no order (exponentials, maxima, the choice of the best k)
// is spread over as many threads as the chip has.
#include <algorithm>
#include <cmath>

#include "xp_device.hpp"
#include "xp_launch.hpp"

namespace xp {

namespace {

constexpr uint32_t kScThreads = 256;
constexpr uint32_t kTopkMax = 64;          // XP_TOPK_MAX, llm_sampling.cl:255
constexpr uint32_t kTopkThreads = 64;      // one wave: 64 x 64 x 8 B = 32 KiB of LDS
constexpr uint32_t kRankTile = 2048;       // candidates staged per LDS tile
constexpr uint32_t kNone = 0xFFFFFFFFu;    // unfilled candidate slot

uint32_t blocks(uint32_t n, uint32_t per) { return (n - 1u) / per + 1u; }   // n > 0

// topk_partial: a wave a chain or a thread a chain, by their times in us
// (measured over 1 to 128 elements, 16 to 262144 chains, k 1 to 64). A thread
// inserts: a chain's elements in turn, each past up to k others, 81920 chains at
// once (a workgroup's lists are 32 KiB of LDS). A wave searches, 1024 elements at
// a time, and takes a chip's share however short its chain, less where the
// chain is no longer than k. Thread / wave: 262144 chains of 16, k = 1 14.4 /
// 256, k = 64 393 / 182; 4096 of 8, k = 1 4.1 / 8.0, k = 8 7.9 / 5.4; 256 of 64,
// k = 8 49.6 / 5.6. A wave a chain stays below a grid's 2^32 threads.
bool topk_by_wave(uint32_t n, uint32_t nparts, uint32_t k) {
    if (nparts >= 1u << 26) return false;
    const double rows = double(n / nparts + (n % nparts != 0u)), p = nparts;
    const double thread = 2.0 + rows * (0.08 + 0.095 * k) * double((nparts - 1u) / 81920u + 1u);
    const double wave = rows <= k ? 3.0 + 0.68e-3 * p : std::max(5.8, 4.8 + 0.98e-3 * p * std::ceil(rows / 1024.0));
    return wave < thread;
}

}  // namespace

__global__ __launch_bounds__(kScThreads) void temperature_kernel(float* x, float inv_temp, uint32_t n) {
    const uint32_t i = blockIdx.x * kScThreads + threadIdx.x;
    if (i < n) x[i] = x[i] * inv_temp;
}

// Chains share a workgroup sixteen at a time: thread t takes chain t % 16 and
// rows t / 16, t / 16 + 16, ... (element p + row * nparts), so a wave's load is
// four 64-byte runs and a chain's elements are worked on by sixteen threads.
// With a thread a chain (a few thousand threads, one load in flight each)
// n = 262144 in 4096 chains took 8.6 us for the maximum and 14.8 for the
// exponentials; now 2.6 and 3.7.
constexpr uint32_t kChainW = 16;                         // chains a workgroup
constexpr uint32_t kChainR = kScThreads / kChainW;       // rows at a time
constexpr uint32_t kChainU = 4;                          // rows in flight a thread

// Short chains, or so many that a thread each fills the chip, need no sharing:
// there the sixteen threads only cost launches of workgroups (and a grid has
// less than 2^32 threads, which 2^28 chains would pass). Tiled / a thread each:
//   maximum      65536 chains of 24  3.9 / 4.1 us, of 64  3.8 / 8.3; 262144 of 4  5.3 / 3.9, of 64  21.7 / 21.6
//   exponentials 65536 chains of 8  5.2 / 4.2, of 24  5.8 / 6.9; 262144 of 1  13.3 / 4.2, of 32  18.1 / 15.3
// From 131072 chains on (512 threads a CU) a thread each has the loads in
// flight; a thread's exponentials are a serial chain besides, which that many
// chains must be long against.
bool max_by_thread(uint32_t n, uint32_t nparts) { return n / nparts < 24u || nparts >= 131072u; }
bool exp_by_thread(uint32_t n, uint32_t nparts) { return n / nparts < 16u || nparts >= 4096u * uint64_t(n / nparts); }

__global__ __launch_bounds__(kScThreads) void reduce_max_partial_thread_kernel(float* pmax, const float* x,
                                                                               uint32_t n, uint32_t nparts) {
    const uint32_t p = blockIdx.x * kScThreads + threadIdx.x;
    if (p >= nparts) return;
    float m = -INFINITY;
    for (uint64_t k = p; k < n; k += nparts) m = fmaxf(m, x[k]);
    pmax[p] = m;
}

__global__ __launch_bounds__(kScThreads) void softmax_exp_partial_thread_kernel(float* out, float* psum, const float* x,
                                                                                const float* stats, uint32_t n,
                                                                                uint32_t nparts) {
    const uint32_t p = blockIdx.x * kScThreads + threadIdx.x;
    if (p >= nparts) return;
    const float m = stats[0];
    float s = 0.0f;
    for (uint64_t k = p; k < n; k += nparts) {
        const float e = expf(x[k] - m);
        out[k] = e;
        s += e;
    }
    psum[p] = s;
}

// The maximum is the same in any order.
__global__ __launch_bounds__(kScThreads) void reduce_max_partial_kernel(float* pmax, const float* x,
                                                                        uint32_t n, uint32_t nparts) {
    __shared__ float sm[kChainR][kChainW];
    const uint32_t c = threadIdx.x % kChainW, r0 = threadIdx.x / kChainW, p = blockIdx.x * kChainW + c;
    float m = -INFINITY;
    if (p < nparts)
        for (uint64_t k = p + uint64_t(r0) * nparts; k < n; k += uint64_t(kChainU * kChainR) * nparts) {
            float v[kChainU];
#pragma unroll
            for (uint32_t u = 0; u < kChainU; ++u) {
                const uint64_t e = k + uint64_t(u * kChainR) * nparts;
                v[u] = e < n ? x[e] : -INFINITY;
            }
#pragma unroll
            for (uint32_t u = 0; u < kChainU; ++u) m = fmaxf(m, v[u]);
        }
    sm[r0][c] = m;
    __syncthreads();
    if (r0 == 0 && p < nparts) {
#pragma unroll
        for (uint32_t r = 1; r < kChainR; ++r) m = fmaxf(m, sm[r][c]);
        pmax[p] = m;
    }
}

// The maximum is the same in any order (fmax drops NaNs either way), so the
// finaliser is a parallel reduction.
__global__ __launch_bounds__(1024) void reduce_max_final_kernel(float* stats, const float* pmax,
                                                                uint32_t nparts) {
    __shared__ float wm[1024 / kWave];
    float m = -INFINITY;
    for (uint32_t p = threadIdx.x; p < nparts; p += 1024) m = fmaxf(m, pmax[p]);
    m = wave_max(m);
    if (threadIdx.x % kWave == 0) wm[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 1024 / kWave; ++w) m = fmaxf(m, wm[w]);
        stats[0] = m;
    }
}

// The exponentials of a 64-row tile by all threads, then each chain's sum in
// chain order by one. `out` may alias `x`: every element is read and written
// by the same thread, its tile's loads before its stores.
__global__ __launch_bounds__(kScThreads) void softmax_exp_partial_kernel(float* out, float* psum,
                                                                         const float* x,
                                                                         const float* stats,
                                                                         uint32_t n, uint32_t nparts) {
    constexpr uint32_t TR = kChainU * kChainR;
    __shared__ float se[TR][kChainW + 1];
    const uint32_t c = threadIdx.x % kChainW, r0 = threadIdx.x / kChainW, p = blockIdx.x * kChainW + c;
    const bool live = p < nparts;
    const float m = stats[0];
    const uint64_t rows = (uint64_t(n) + nparts - 1u) / nparts;   // of the longest chain
    float s = 0.0f;
    for (uint64_t t = 0; t < rows; t += TR) {
        float v[kChainU];
#pragma unroll
        for (uint32_t u = 0; u < kChainU; ++u) {
            const uint64_t e = p + (t + r0 + u * kChainR) * nparts;
            v[u] = live && e < n ? x[e] : 0.0f;
        }
#pragma unroll
        for (uint32_t u = 0; u < kChainU; ++u) {
            const uint64_t e = p + (t + r0 + u * kChainR) * nparts;
            const float g = expf(v[u] - m);
            if (live && e < n) out[e] = g;
            se[r0 + u * kChainR][c] = g;
        }
        __syncthreads();
        if (r0 == 0 && live && p < n) {
            const uint64_t mine = (uint64_t(n) - p + nparts - 1u) / nparts;   // this chain's rows
            const uint32_t left = uint32_t(mine > t ? (mine - t < TR ? mine - t : TR) : 0u);
            if (left == TR) {
#pragma unroll
                for (uint32_t r = 0; r < TR; ++r) s += se[r][c];
            } else {
                for (uint32_t r = 0; r < left; ++r) s += se[r][c];
            }
        }
        __syncthreads();
    }
    if (r0 == 0 && live) psum[p] = s;
}

__global__ __launch_bounds__(kScThreads) void reduce_sum_partial_kernel(float* out, const float* in,
                                                                        uint32_t n, uint32_t nparts) {
    const uint32_t p = blockIdx.x * kScThreads + threadIdx.x;
    if (p >= nparts) return;
    float s = 0.0f;
    for (uint32_t k = p; k < n; k += nparts) s += in[k];
    out[p] = s;
}

// ---- serial sums ------------------------------------------------------------
// The reference adds in one order, and the fp32 sum depends on it. A lone chain
// of dependent adds costs 8 cycles each (15 us for 4096), but where the running
// sum s keeps its exponent, adding v >= 0 adds the whole number rint(v / u) of
// s's last places u, whatever the terms before it: only a tie (v / u halfway
// between two whole numbers) looks at s, at its last bit. So a wave adds a
// block at once, as whole numbers below 2^24, and gets the serial sum bit for bit.
// A block in which the exponent would change, or with a term that is negative,
// not finite or more than a quarter of s, is refused and added one by one.
__device__ __forceinline__ bool sum_scale(float s, int& sh) {
    const uint32_t e = __float_as_uint(s) >> 23;
    sh = 150 - int(e);                                   // v / u = v 2^sh
    return e - 1u < 254u;                                // positive, normal, finite
}
// s + the last places `more`, if that keeps the exponent.
__device__ __forceinline__ bool sum_grow(float& s, float more, uint32_t ties) {
    const uint32_t b = __float_as_uint(s);
    if (!(more + float(ties) < 8388608.0f - float(b & 0x7FFFFFu))) return false;
    s = __uint_as_float(b + uint32_t(more) + ties);
    return true;
}
// 256 terms, four a lane in any order; ties are refused.
__device__ __forceinline__ bool sum_block4(float& s, float4 v) {
    int sh;
    if (!sum_scale(s, sh)) return false;
    const float t[4] = {v.x, v.y, v.z, v.w};
    bool ok = true;
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float r = __builtin_amdgcn_ldexpf(t[i], sh), k = __builtin_rintf(r);
        ok = ok && r >= 0.0f && r < 4194304.0f && fabsf(r - k) != 0.5f;
        q += k;                                          // exact: at most 2^24
    }
    if (__ballot(!ok) != 0ull) return false;
    return sum_grow(s, wave_sum(q), 0u);                 // a sum past 2^24 may round, but not to below it
}
// 64 terms, one a lane in order.
__device__ __forceinline__ bool sum_block(float& s, float v) {
    int sh;
    if (!sum_scale(s, sh)) return false;
    const float r = __builtin_amdgcn_ldexpf(v, sh), w = floorf(r), f = r - w;
    if (__ballot(!(r >= 0.0f && r < 4194304.0f)) != 0ull) return false;
    const float k = w + (f > 0.5f ? 1.0f : 0.0f);
    unsigned long long tie = __ballot(f == 0.5f);
    uint32_t up = 0;
    if (tie != 0ull) {
        const unsigned long long odd = __ballot((uint32_t(k) & 1u) != 0u);
        for (; tie != 0ull; tie &= tie - 1u) {           // to even: up where the sum before it, and its whole part, are odd
            const int i = __builtin_ctzll(tie);
            up += (__float_as_uint(s) + uint32_t(__builtin_popcountll(odd & ((2ull << i) - 1ull))) + up) & 1u;
        }
    }
    return sum_grow(s, wave_sum(k), up);
}

constexpr uint32_t kSerTile = 4096, kSerBlock = 256;
static_assert(kSerTile % kSerBlock == 0, "whole blocks");
// A tile of terms to LDS by all threads, zeros up to a whole block (s + 0 is s).
__device__ __forceinline__ uint32_t serial_tile(float* tile, const float* src, uint32_t base, uint32_t n) {
    const uint32_t m = min(kSerTile, n - base);
    for (uint32_t i = threadIdx.x; i < (m + kSerBlock - 1u) / kSerBlock * kSerBlock; i += kScThreads) tile[i] = i < m ? src[base + i] : 0.0f;
    __syncthreads();
    return m;
}
__device__ __forceinline__ void ld16(float (&v)[16], const float* p) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 q = *reinterpret_cast<const float4*>(p + 4 * i);
        v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
    }
}

// 4096 sums: 64 us by one thread from memory, 18.6 as a chain of adds from
// LDS, 16.1 in blocks.
__global__ __launch_bounds__(kScThreads) void reduce_sum_final_kernel(float* stats, const float* psum, uint32_t nparts) {
    __shared__ __attribute__((aligned(16))) float tile[kSerTile];
    float s = 0.0f;
    for (uint32_t base = 0; base < nparts; base += kSerTile) {
        __syncthreads();
        const uint32_t m = serial_tile(tile, psum, base, nparts);
        if (threadIdx.x < kWave) {
            for (uint32_t i = 0; i < m; i += kSerBlock) {
                if (sum_block4(s, *reinterpret_cast<const float4*>(tile + i + 4u * threadIdx.x))) continue;
                for (uint32_t j = i; j < i + kSerBlock; j += kWave) {
                    if (sum_block(s, tile[j + threadIdx.x])) continue;
                    for (uint32_t h = j; h < j + kWave; h += 16) {
                        float v[16];
                        ld16(v, tile + h);
#pragma unroll
                        for (int x = 0; x < 16; ++x) s += v[x];
                    }
                }
            }
        }
    }
    if (threadIdx.x == 0) stats[1] = s;
}

__global__ __launch_bounds__(kScThreads) void softmax_normalize_kernel(float* out, const float* stats,
                                                                       uint32_t n) {
    const uint32_t i = blockIdx.x * kScThreads + threadIdx.x;
    if (i < n) out[i] = out[i] / stats[1];
}

// Chain p's best k (descending, strict '>' so the earliest index wins a tie),
// unfilled slots (-inf, none). bv / bi are [slot][thread] in LDS.
__global__ __launch_bounds__(kTopkThreads) void topk_partial_kernel(float* cval, uint32_t* cidx,
                                                                    const float* x, uint32_t n,
                                                                    uint32_t nparts, uint32_t k) {
    __shared__ float bv[kTopkMax][kTopkThreads];
    __shared__ uint32_t bi[kTopkMax][kTopkThreads];
    x += size_t(blockIdx.y) * n;                       // batched rows (grid.y)
    cval += size_t(blockIdx.y) * nparts * k;
    cidx += size_t(blockIdx.y) * nparts * k;
    const uint32_t t = threadIdx.x;
    const uint32_t p = blockIdx.x * kTopkThreads + t;
    for (uint32_t j = 0; j < k; ++j) { bv[j][t] = -INFINITY; bi[j][t] = kNone; }
    if (p >= nparts) return;
    float thr = -INFINITY;                       // bv[k - 1][t]
    for (uint64_t e = p; e < n; e += nparts) {
        const float v = x[e];
        if (!(v > thr)) continue;
        uint32_t j = k - 1u;
        while (j > 0u && v > bv[j - 1u][t]) {
            bv[j][t] = bv[j - 1u][t];
            bi[j][t] = bi[j - 1u][t];
            --j;
        }
        bv[j][t] = v;
        bi[j][t] = uint32_t(e);
        thr = bv[k - 1u][t];
    }
    for (uint32_t j = 0; j < k; ++j) {
        cval[size_t(p) * k + j] = bv[j][t];
        cidx[size_t(p) * k + j] = bi[j][t];
    }
}

// ---- exact best k (<= 64) of a wave's values --------------------------------
// Values live in registers, R a lane, with an order-preserving key (0 = no
// candidate) and an id; the best k by (value desc, id asc) are found without
// sorting: the k-th largest key bit by bit from the top, each bit one count
// over the wave (R compares and ballots), starting below the bits that the
// largest and the smallest lane maximum share (at least 64 keys reach the
// latter) and ending as soon as a cut keeps exactly k; only a tie across the
// cut is resolved further, by id. A thread inserting element by element into
// its own sorted list in LDS took 5.1 ms for 256 chains of 1024 and k = 64,
// this 11 us.
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ uint32_t value_key(float v) { return order_key(v + 0.0f); }   // -0 ties with 0

template <int R>
__device__ __forceinline__ uint32_t count_ge(const uint32_t (&key)[R], uint32_t t) {
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) c += uint32_t(__popcll(__ballot(key[j] >= t)));
    return c;
}
__device__ __forceinline__ uint32_t lanes_below(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
}
// LDS written by some lanes of a wave is read by others of it: in order in
// the hardware, kept in order in the code.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Bits b and below of the k-th largest key, from the top, into t: until the
// cut keeps at most `enough`. cnt keys reach t.
template <int R>
__device__ __forceinline__ int search_cut(const uint32_t (&key)[R], uint32_t k, uint32_t enough, int b, uint32_t& t, uint32_t& cnt) {
    for (; b >= 0 && cnt > enough; --b) {
        const uint32_t c = count_ge(key, t | (1u << b));
        if (c >= k) {
            t |= 1u << b;
            cnt = c;
        }
    }
    return b;
}
// The survivors (at most k, in no order) to sv / si; returns their number.
// cnt keys reach t, which has the k-th largest key's bits above b.
template <int R>
__device__ __forceinline__ uint32_t wave_cut(const float (&v)[R], const uint32_t (&id)[R], const uint32_t (&key)[R],
                                             uint32_t k, int bit, uint32_t t, uint32_t cnt, float* sv, uint32_t* si) {
    uint32_t tie_id = kNone;
    bool ties = false;
    if (cnt > k) {
        search_cut(key, k, k, bit, t, cnt);
        if (cnt > k) {   // the k-th largest key is t, with more of it than fit
            ties = true;
            uint32_t g = 0;
#pragma unroll
            for (int j = 0; j < R; ++j) g += uint32_t(__popcll(__ballot(key[j] > t)));
            tie_id = 0u;
            for (int b = 31; b >= 0; --b) {
                const uint32_t u = tie_id | ((1u << b) - 1u);
                uint32_t c = 0;
#pragma unroll
                for (int j = 0; j < R; ++j) c += uint32_t(__popcll(__ballot(key[j] == t && id[j] <= u)));
                if (c < k - g) tie_id |= 1u << b;
            }
        }
    }
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const bool take = ties ? key[j] > t : key[j] >= t;
        const unsigned long long b = __ballot(take);
        const uint32_t at = m + lanes_below(b);
        if (take) {
            sv[at] = v[j];
            si[at] = id[j];
        }
        m += uint32_t(__popcll(b));
    }
    if (ties) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const bool take = key[j] == t && id[j] <= tie_id;
            const unsigned long long b = __ballot(take);
            const uint32_t at = m + lanes_below(b);
            if (take && at < k) {
                sv[at] = v[j];
                si[at] = id[j];
            }
            m = min(k, m + uint32_t(__popcll(b)));
        }
    }
    wave_lds_sync();
    return m;
}

// A search over 17 registers a lane is 51 instructions a bit: once the cut
// keeps kBestFew, those move to LDS and back to five registers a lane.
constexpr int kFewR = 5;
constexpr uint32_t kBestFew = kFewR * kWave;
struct BestFew {
    float v[kBestFew];
    uint32_t id[kBestFew];
};
template <int R>
__device__ __forceinline__ uint32_t wave_best(const float (&v)[R], const uint32_t (&id)[R], const uint32_t (&key)[R],
                                              uint32_t k, BestFew& few, float* sv, uint32_t* si) {
    uint32_t t = 1u, cnt = count_ge(key, 1u);
    int bit = -1;
    if (cnt > k) {
        uint32_t lm = 0;
#pragma unroll
        for (int j = 0; j < R; ++j) lm = max(lm, key[j]);
        uint32_t hi = lm, lo = lm;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            hi = max(hi, uint32_t(__shfl_xor(int(hi), o, kWave)));
            lo = min(lo, uint32_t(__shfl_xor(int(lo), o, kWave)));
        }
        hi = __builtin_amdgcn_readfirstlane(hi);
        lo = __builtin_amdgcn_readfirstlane(lo);
        const int nb = hi == lo ? 0 : 32 - __builtin_clz(hi ^ lo);
        t = nb >= 32 ? 0u : hi & ~((1u << nb) - 1u);
        cnt = t == 0u ? 0xFFFFFFFFu : count_ge(key, t);
        bit = search_cut(key, k, max(k, kBestFew), nb - 1, t, cnt);
    }
    if (cnt > kBestFew) return wave_cut(v, id, key, k, bit, t, cnt, sv, si);   // that many equal keys
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const bool take = key[j] >= t;
        const unsigned long long b = __ballot(take);
        const uint32_t at = m + lanes_below(b);
        if (take) {
            few.v[at] = v[j];
            few.id[at] = id[j];
        }
        m += uint32_t(__popcll(b));
    }
    wave_lds_sync();
    const uint32_t lane = threadIdx.x % kWave;
    float fv[kFewR];
    uint32_t fid[kFewR], fkey[kFewR];
#pragma unroll
    for (int j = 0; j < kFewR; ++j) {
        const uint32_t at = uint32_t(j) * kWave + lane;
        fv[j] = few.v[at];
        fid[j] = at < m ? few.id[at] : kNone;
        fkey[j] = at < m ? value_key(fv[j]) : 0u;
    }
    wave_lds_sync();
    return wave_cut(fv, fid, fkey, k, bit, t, cnt, sv, si);
}

// Lane i < m of a wave's m survivors: its value, id and rank, the number of
// survivors that beat it. The slots past m are filled with what beats nothing.
__device__ __forceinline__ uint32_t wave_rank(float* sv, uint32_t* si, uint32_t m, float& v, uint32_t& d) {
    const uint32_t lane = threadIdx.x % kWave;
    if (lane >= m) {
        sv[lane] = -INFINITY;
        si[lane] = kNone;
    }
    wave_lds_sync();
    v = sv[lane];
    d = si[lane];
    uint32_t rank = 0;
    for (uint32_t j = 0; j < m; j += 8) {
        float w[8];
        uint32_t e[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
            w[i] = sv[j + i];
            e[i] = si[j + i];
        }
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) rank += (w[i] > v) | ((w[i] == v) & (e[i] < d));
    }
    return rank;
}

constexpr int kBestR = 17;                               // the survivors so far, and 16 new values a lane

// Chain p's best k (descending, the earliest index first among equals),
// unfilled slots (-inf, none): one wave a chain, 1024 elements at a time.
__global__ __launch_bounds__(kWave) void topk_partial_wave_kernel(float* cval, uint32_t* cidx, const float* x,
                                                                 uint32_t n, uint32_t nparts, uint32_t k) {
    __shared__ __attribute__((aligned(16))) float sv[kTopkMax];
    __shared__ __attribute__((aligned(16))) uint32_t si[kTopkMax];
    __shared__ BestFew few;
    const uint32_t p = blockIdx.x, lane = threadIdx.x;
    uint32_t m = 0;
    for (uint64_t r0 = 0; p + r0 * nparts < n; r0 += 1024u) {
        float v[kBestR];
        uint32_t id[kBestR], key[kBestR];
        v[0] = lane < m ? sv[lane] : 0.0f;
        id[0] = lane < m ? si[lane] : kNone;
        key[0] = lane < m ? value_key(v[0]) : 0u;
#pragma unroll
        for (int j = 1; j < kBestR; ++j) {
            const uint64_t e = p + (r0 + uint32_t(j - 1) * kWave + lane) * nparts;
            id[j] = uint32_t(e);
            v[j] = e < n ? x[e] : -INFINITY;
        }
#pragma unroll
        for (int j = 1; j < kBestR; ++j) key[j] = v[j] > -INFINITY ? value_key(v[j]) : 0u;   // no NaN either
        wave_lds_sync();                                 // slot 0 is read before it is written
        m = wave_best(v, id, key, k, few, sv, si);
    }
    float v = -INFINITY;
    uint32_t d = kNone, rank = lane;
    if (m > 0) {
        float wv;
        uint32_t wd;
        const uint32_t wr = wave_rank(sv, si, m, wv, wd);
        if (lane < m) {
            v = wv;
            d = wd;
            rank = wr;
        }
    }
    if (rank < k) {                                      // lanes past m fill the slots past the survivors
        cval[size_t(p) * k + rank] = v;
        cidx[size_t(p) * k + rank] = d;
    }
}

// The best k <= 64 of a candidate list by (value desc, index asc) to oval /
// oidx[rank], one workgroup: each wave keeps the best k of its share, the
// first wave the best of those. Slots with no candidate of that rank are not
// written. Counting every candidate against every other took 512 us for 16384; this
// takes 14.5 (17 where every bit was a count over all registers).
__global__ __launch_bounds__(1024) void topk_rank_wave_kernel(float* oval, uint32_t* oidx, const float* cval,
                                                             const uint32_t* cidx, uint32_t ncand, uint32_t k) {
    __shared__ __attribute__((aligned(16))) float sv[16][kTopkMax];
    __shared__ __attribute__((aligned(16))) uint32_t si[16][kTopkMax];
    __shared__ BestFew few[16];
    __shared__ uint32_t sm[16];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const uint32_t waves = blockDim.x / kWave;
    uint32_t m = 0;
    for (uint64_t b = uint64_t(wave) * 1024u; b < ncand; b += uint64_t(waves) * 1024u) {
        float v[kBestR];
        uint32_t id[kBestR], key[kBestR];
        v[0] = lane < m ? sv[wave][lane] : 0.0f;
        id[0] = lane < m ? si[wave][lane] : kNone;
        key[0] = lane < m ? value_key(v[0]) : 0u;
#pragma unroll
        for (int j = 1; j < kBestR; ++j) {
            const uint64_t i = b + uint32_t(j - 1) * kWave + lane;
            v[j] = i < ncand ? cval[i] : 0.0f;
            id[j] = i < ncand ? cidx[i] : kNone;
        }
#pragma unroll
        for (int j = 1; j < kBestR; ++j) {
            if (id[j] != kNone && v[j] != v[j]) {        // beaten by none and beating none: rank 0, as ever
                oval[0] = v[j];
                oidx[0] = id[j];
            }
            key[j] = id[j] != kNone && v[j] == v[j] ? value_key(v[j]) : 0u;
        }
        wave_lds_sync();
        m = wave_best(v, id, key, k, few[wave], sv[wave], si[wave]);
    }
    if (waves > 1) {
        if (lane == 0) sm[wave] = m;
        __syncthreads();
        if (wave != 0) return;
        float v[kBestR];
        uint32_t id[kBestR], key[kBestR];
        v[0] = 0.0f;
        id[0] = kNone;
        key[0] = 0u;
#pragma unroll
        for (int j = 1; j < kBestR; ++j) {
            const bool in = uint32_t(j - 1) < waves && lane < sm[j - 1];
            v[j] = in ? sv[j - 1][lane] : 0.0f;
            id[j] = in ? si[j - 1][lane] : kNone;
            key[j] = in ? value_key(v[j]) : 0u;
        }
        wave_lds_sync();
        m = wave_best(v, id, key, k, few[0], sv[0], si[0]);
    }
    if (wave != 0 || m == 0) return;
    float v;
    uint32_t d;
    const uint32_t rank = wave_rank(sv[0], si[0], m, v, d);
    if (lane < m) {
        oval[rank] = v;
        oidx[rank] = d;
    }
}

// Candidate i's rank = number of filled candidates beating it by (value
// desc, index asc); rank < k writes out[rank]. Candidates pass through LDS in
// tiles that every thread of the workgroup scans.
__global__ __launch_bounds__(kScThreads) void topk_rank_select_kernel(float* oval, uint32_t* oidx,
                                                                      const float* cval,
                                                                      const uint32_t* cidx,
                                                                      uint32_t ncand, uint32_t k) {
    __shared__ float tv[kRankTile];
    __shared__ uint32_t ti[kRankTile];
    cval += size_t(blockIdx.y) * ncand;                 // batched rows (grid.y)
    cidx += size_t(blockIdx.y) * ncand;
    oval += size_t(blockIdx.y) * k;
    oidx += size_t(blockIdx.y) * k;
    const uint32_t i = blockIdx.x * kScThreads + threadIdx.x;
    const bool mine = i < ncand;
    const float v = mine ? cval[i] : -INFINITY;
    const uint32_t d = mine ? cidx[i] : kNone;
    uint32_t rank = 0;
    for (uint32_t base = 0; base < ncand; base += kRankTile) {
        const uint32_t m = min(kRankTile, ncand - base);
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < m; j += kScThreads) {
            tv[j] = cval[base + j];
            ti[j] = cidx[base + j];
        }
        __syncthreads();
        for (uint32_t j = 0; j < m; ++j) {
            const float w = tv[j];
            const uint32_t e = ti[j];
            rank += (e != kNone) & ((w > v) | ((w == v) & (e < d)));
        }
    }
    if (mine && d != kNone && rank < k) {
        oval[rank] = v;
        oidx[rank] = d;
    }
}

__global__ __launch_bounds__(kScThreads) void topk_mask_kernel(float* logits, const float* topk_val,
                                                               uint32_t k, uint32_t n) {
    const uint32_t i = blockIdx.x * kScThreads + threadIdx.x;
    if (i >= n) return;
    const float t = topk_val[k - 1u];
    if (logits[i] < t) logits[i] = -INFINITY;
}

// Serial over k (the reference's top-p is a single work-item): a wave brings
// 256 weights at a time to LDS (zeros past the end) and every lane adds them in
// order, sixteen read at once.
constexpr uint32_t kDrawTile = 256;
__device__ __forceinline__ float lane_f(float v, uint32_t l) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), int(l)));
}
__device__ __forceinline__ void draw_tile(float* tile, const float* w, uint32_t b, uint32_t k) {
    wave_lds_sync();
#pragma unroll
    for (uint32_t j = 0; j < kDrawTile; j += kWave)
        tile[j + threadIdx.x] = b + j + threadIdx.x < k ? w[b + j + threadIdx.x] : 0.0f;
    wave_lds_sync();
}
__device__ __forceinline__ float serial_total(float* tile, const float* w, uint32_t k) {
    float total = 0.0f;
    for (uint32_t b = 0; b < k; b += kDrawTile) {
        draw_tile(tile, w, b, k);
        for (uint32_t i = 0; i < kDrawTile && b + i < k; i += 16) {
            float v[16];
            ld16(v, tile + i);
#pragma unroll
            for (int j = 0; j < 16; ++j) total += v[j];
        }
    }
    return total;
}

__global__ __launch_bounds__(kWave) void topp_cutoff_kernel(float* w, uint32_t k, float p) {
    __shared__ __attribute__((aligned(16))) float tile[kDrawTile];
    const float total = serial_total(tile, w, k);
    if (!(total > 0.0f)) return;
    // every weight from the first whose running mass before it reaches the
    // cut on: past it the mass no longer grows
    const float cut = p * total;
    float cum = 0.0f;
    uint32_t keep = kNone;
    for (uint32_t b = 0; b < k && keep == kNone; b += kDrawTile) {
        draw_tile(tile, w, b, k);
        for (uint32_t i = 0; i < kDrawTile && b + i < k && keep == kNone; i += 16) {
            float v[16];
            ld16(v, tile + i);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                if (keep == kNone && cum >= cut) keep = b + i + j;
                cum += v[j];
            }
        }
    }
    if (keep == kNone) return;
    for (uint64_t j = uint64_t(keep) + threadIdx.x; j < k; j += kWave) w[j] = 0.0f;
}

__global__ __launch_bounds__(kWave) void multinomial_sample_kernel(float* out, uint32_t* idx_out, const float* w,
                                                                   const uint32_t* idx, uint32_t k, float u) {
    __shared__ __attribute__((aligned(16))) float tile[kDrawTile];
    const float target = u * serial_total(tile, w, k);
    float cum = 0.0f, cw = 0.0f;
    uint32_t at = kNone;                                 // the last weight above zero up to the stop
    bool stop = false;
    for (uint32_t b = 0; b < k && !stop; b += kDrawTile) {
        draw_tile(tile, w, b, k);
        for (uint32_t i = 0; i < kDrawTile && b + i < k && !stop; i += 16) {
            float v[16];
            ld16(v, tile + i);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                if (!stop && v[j] > 0.0f) {
                    at = b + i + j;
                    cw = v[j];
                }
                cum += v[j];
                stop = stop || cum > target;
            }
        }
    }
    if (threadIdx.x != 0) return;
    const uint32_t chosen = at == kNone ? 0u : idx[at];
    out[0] = float(chosen);
    out[1] = cw;
    idx_out[0] = chosen;
}

// The chain whose running mass passes the target, then the element in it: the
// sums and their order are the reference's, from LDS tiles in blocks as in
// reduce_sum_final (4096 chains of 64: 250 us by one thread, 31.5 as a chain of adds,
// 19 so). A block added at once has no negative term: it is passed over where
// its end has not passed the target. In one that may hold the place, sixteen
// running sums are formed before their largest is held against the target.
__global__ __launch_bounds__(kScThreads) void multinomial_strided_kernel(float* out, uint32_t* idx_out, const float* w,
                                                                         const float* psum, const float* stats,
                                                                         uint32_t n, uint32_t nparts, float u) {
    __shared__ __attribute__((aligned(16))) float tile[kSerTile];
    __shared__ uint32_t found;
    const float target = u * stats[1];
    float cum = 0.0f;
    uint32_t chain = kNone;
    if (threadIdx.x == 0) found = 0u;
    for (uint32_t base = 0; base < nparts; base += kSerTile) {
        __syncthreads();
        if (found) break;
        const uint32_t m = serial_tile(tile, psum, base, nparts);
        if (threadIdx.x < kWave) {
            // sixteen running sums; true once one has passed the target
            auto step = [&](const float (&v)[16], uint32_t at) {
                float c[16];
                c[0] = cum + v[0];
#pragma unroll
                for (int j = 1; j < 16; ++j) c[j] = c[j - 1] + v[j];
                float mx = c[0];
#pragma unroll
                for (int j = 1; j < 16; ++j) mx = fmaxf(mx, c[j]);
                if (!(mx > target)) {
                    cum = c[15];
                    return false;
                }
                uint32_t f = 0;
#pragma unroll
                for (int j = 15; j >= 0; --j)
                    if (c[j] > target) f = uint32_t(j);
                // the running sum is not added past the chosen chain
#pragma unroll
                for (int j = 0; j < 15; ++j)
                    if (f == uint32_t(j) + 1u) cum = c[j];
                chain = base + at + f;
                return true;
            };
            for (uint32_t i = 0; i < m && chain == kNone; i += kSerBlock) {
                float c = cum;
                if (sum_block4(c, *reinterpret_cast<const float4*>(tile + i + 4u * threadIdx.x)) && !(c > target)) {
                    cum = c;
                    continue;
                }
                for (uint32_t j = i; j < i + kSerBlock && chain == kNone; j += kWave) {
                    c = cum;
                    if (sum_block(c, tile[j + threadIdx.x]) && !(c > target)) {
                        cum = c;
                        continue;
                    }
                    for (uint32_t h = j; h < j + kWave; h += 16) {
                        float v[16];
                        ld16(v, tile + h);
                        if (step(v, h)) break;
                    }
                }
            }
            if (threadIdx.x == 0 && chain != kNone) found = 1u;
        }
    }
    if (threadIdx.x >= kWave) return;
    if (chain == kNone) chain = nparts - 1u;
    // The element, 64 of the chain at a time, as the chain was found: sixteen
    // running sums from LDS (with zeros past the chain's end, which pass no
    // target that the last element did not), 12 ns an element on a chain of
    // 32768; up to sixteen elements one by one from the lanes, which waits for
    // no LDS (60 ns an element). The last element if none passes.
    uint32_t chosen = chain;
    float cw = 0.0f;
    for (uint64_t b = chain; b < n; b += uint64_t(kWave) * nparts) {
        const uint64_t e = b + uint64_t(threadIdx.x) * nparts;
        const float v = e < n ? w[e] : 0.0f;
        const uint64_t left = (uint64_t(n) - b + nparts - 1u) / nparts;
        uint32_t at = uint32_t(left < kWave ? left : kWave) - 1u;
        bool stop = false;
        if (at < 16u) {
            for (uint32_t j = 0, last = at; j <= last && !stop; ++j) {
                at = j;
                cum += lane_f(v, j);
                stop = cum > target;
            }
            cw = lane_f(v, at);
        } else {
            wave_lds_sync();
            tile[threadIdx.x] = v;
            wave_lds_sync();
            for (uint32_t h = 0; h <= at && !stop; h += 16) {
                float x[16], c[16];
                ld16(x, tile + h);
                c[0] = cum + x[0];
#pragma unroll
                for (int j = 1; j < 16; ++j) c[j] = c[j - 1] + x[j];
                float mx = c[0];
#pragma unroll
                for (int j = 1; j < 16; ++j) mx = fmaxf(mx, c[j]);
                cum = c[15];                             // not used again once one has passed
                if (!(mx > target)) continue;
#pragma unroll
                for (int j = 15; j >= 0; --j)
                    if (c[j] > target) {
                        at = h + uint32_t(j);
                        stop = true;
                    }
            }
            cw = tile[at];
        }
        chosen = uint32_t(b + uint64_t(at) * nparts);
        if (stop) break;
    }
    if (threadIdx.x != 0) return;
    out[0] = float(chosen);
    out[1] = cw;
    idx_out[0] = chosen;
}

// Exact best k of a candidate list, one workgroup per row: a most-significant-
// byte-first radix select finds the k-th largest (value, as an order-preserving
// key); the candidates at or above it (k plus any ties) are gathered in LDS and
// ranked among themselves by (value desc, index asc). Exact while fewer than
// 256 - k candidates tie with the k-th largest value. Logits share their top
// bytes, so most of a wave's keys fall in one bin: the histogram is kept in
// kSelCopies copies, lane l adding to copy l % kSelCopies (a bin's copies in
// consecutive words, different banks), which turns a 64-way same-address
// atomic into a 4-way one, and each thread adds a run of its keys that fall
// in one bin with one atomic; the copies are summed before the scan.
constexpr uint32_t kSelThreads = 1024;
constexpr uint32_t kSelPer = 16;             // candidates per thread (16384 per row)
constexpr uint32_t kSelKeep = 256;           // survivors ranked (k + ties)
static_assert(kTopkMax <= kSelKeep, "the ranked output fits the survivors' slots");
constexpr uint32_t kSelCopies = 16;          // histogram copies
constexpr uint32_t kSelStride = kSelCopies + 1u;   // words per bin (padded: the sum reads bins apart)

__global__ __launch_bounds__(kSelThreads) void select_rows_kernel(float* oval, uint32_t* oidx,
                                                                  const float* cval,
                                                                  const uint32_t* cidx,
                                                                  uint32_t ncand, uint32_t k,
                                                                  uint32_t* pos_inc) {
    __shared__ uint32_t hcopy[256 * kSelStride];
    __shared__ uint32_t hist[256];
    __shared__ uint32_t sel[3];               // prefix, needed, survivors
    __shared__ float sv[kSelKeep];
    __shared__ uint32_t si[kSelKeep];
    // the ranked output, written to oval / oidx once per slot at the end
    // (the outputs may be host memory, where two stores to one slot from
    // different waves need not land in order)
    __shared__ float ov[kSelKeep];
    __shared__ uint32_t oi[kSelKeep];
    const uint32_t r = blockIdx.x, tid = threadIdx.x;
    cval += size_t(r) * ncand;
    cidx += size_t(r) * ncand;
    if (tid < k) {   // slots no candidate reaches stay unfilled
        ov[tid] = -INFINITY;
        oi[tid] = kNone;
    }
    if (pos_inc && tid == 0) pos_inc[r] += 1u;
    // every candidate's value and index loaded at once (unconditionally, an
    // index past the end reads candidate 0), kept in registers for the gather
    uint32_t key[kSelPer], ci[kSelPer];
    float cv[kSelPer];
#pragma unroll
    for (uint32_t j = 0; j < kSelPer; ++j) {
        const uint32_t i = tid + j * kSelThreads;
        const uint32_t ic = i < ncand ? i : 0u;
        cv[j] = cval[ic];
        ci[j] = cidx[ic];
    }
#pragma unroll
    for (uint32_t j = 0; j < kSelPer; ++j) {
        const uint32_t i = tid + j * kSelThreads;
        key[j] = (i < ncand && ci[j] != kNone) ? order_key(cv[j]) : 0u;   // 0: below every value
    }
    uint32_t prefix = 0, mask = 0, need = k;
    const uint32_t copy = tid % kSelCopies;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (uint32_t i = tid; i < 256u * kSelStride; i += kSelThreads) hcopy[i] = 0;
        __syncthreads();
        {   // a thread's run of keys in one bin goes in with one atomic
            uint32_t rb = 0u, rn = 0u;
#pragma unroll
            for (uint32_t j = 0; j < kSelPer; ++j) {
                if (key[j] != 0u && (key[j] & mask) == prefix) {
                    const uint32_t bin = (key[j] >> shift) & 255u;
                    if (bin != rb) {
                        if (rn) atomicAdd(&hcopy[rb * kSelStride + copy], rn);
                        rb = bin;
                        rn = 0u;
                    }
                    ++rn;
                }
            }
            if (rn) atomicAdd(&hcopy[rb * kSelStride + copy], rn);
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t c = 0;
#pragma unroll
            for (uint32_t q = 0; q < kSelCopies; ++q) c += hcopy[tid * kSelStride + q];
            hist[tid] = c;
        }
        __syncthreads();
        if (tid < kWave) {
            // lane l covers bins 255 - 4 l .. 252 - 4 l; inclusive prefix of
            // the lane counts from the top bin down, then the crossing lane
            // walks its own four bins
            const uint32_t l = tid;
            const uint32_t c0 = hist[255 - 4 * l], c1 = hist[254 - 4 * l], c2 = hist[253 - 4 * l],
                           c3 = hist[252 - 4 * l];
            const uint32_t mine = c0 + c1 + c2 + c3;
            uint32_t incl = mine;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t t = __shfl_up(incl, o, kWave);
                if (l >= uint32_t(o)) incl += t;
            }
            const uint32_t excl = incl - mine;
            if (excl < need && incl >= need) {   // exactly one lane
                uint32_t acc = excl, d = 255 - 4 * l;
                const uint32_t cs[4] = {c0, c1, c2, c3};
                for (int j = 0; j < 4; ++j) {
                    if (acc + cs[j] >= need) { d = 255 - 4 * l - j; break; }
                    acc += cs[j];
                }
                sel[0] = prefix | (d << shift);
                sel[1] = need - acc;
            }
            if (l == kWave - 1 && incl < need) {   // fewer than need keys: keep them all
                sel[0] = prefix;
                sel[1] = need;
            }
        }
        __syncthreads();
        prefix = sel[0];
        need = sel[1];
        mask |= 255u << shift;
        __syncthreads();
    }
    // prefix = the k-th largest key (or 0 when fewer than k candidates exist)
    if (tid == 0) sel[2] = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kSelPer; ++j) {
        if (key[j] != 0u && key[j] >= prefix) {
            const uint32_t slot = atomicAdd(&sel[2], 1u);
            if (slot < kSelKeep) { sv[slot] = cv[j]; si[slot] = ci[j]; }
        }
    }
    __syncthreads();
    const uint32_t m = min(sel[2], kSelKeep);
    if (tid < m) {
        const float v = sv[tid];
        const uint32_t d = si[tid];
        uint32_t rank = 0;
        for (uint32_t j = 0; j < m; ++j) rank += (sv[j] > v) | ((sv[j] == v) & (si[j] < d));
        if (rank < k) {
            ov[rank] = v;
            oi[rank] = d;
        }
    }
    __syncthreads();
    if (tid < k) {
        oval[size_t(r) * k + tid] = ov[tid];
        oidx[size_t(r) * k + tid] = oi[tid];
    }
}

// The sample-first draw of a batched step on the device, one wave per
// sequence, in the host draw's arithmetic (session.cpp draw(), after
// decode.cpp:1893-1915), so that steps can follow each other with no host
// round trip: the candidates are select_rows' output, already in the host
// draw's (value desc, index asc) order; e = exp((v - max) / T) in float (the
// exponential in double, rounded once); the sums, the top-p cut and the
// inverse-CDF walk in double, in candidate order, on one lane; u from
// Philox4x32-10 (Salmon et al. 2011) at (seed, seq0 + row, step), 53 bits.
// Greedy (mode 0) takes candidate 0. Writes the token to tok[row] and to
// hist[(steps[row] % hist_cap) * rows + row], and advances steps[row] (in
// greedy mode a history counter only).
__device__ __forceinline__ void philox4x32_10_dev(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                  uint32_t k0, uint32_t k1, uint32_t (&o)[4]) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        const uint32_t hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
        const uint32_t hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
        const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
    }
    o[0] = c0;
    o[1] = c1;
    o[2] = c2;
    o[3] = c3;
}

__global__ __launch_bounds__(kWave) void draw_rows_kernel(const float* val, const uint32_t* idx, uint32_t k,
                                                          int mode, float temperature, uint32_t top_k,
                                                          float top_p, uint32_t seed, uint32_t seq0,
                                                          uint32_t* steps, uint32_t* tok, uint32_t* hist,
                                                          uint32_t hist_cap) {
    __shared__ float sv[kWave], se[kWave];
    __shared__ uint32_t si[kWave];
    const uint32_t row = blockIdx.x, lane = threadIdx.x, rows = gridDim.x;
    if (mode == 0) {
        if (lane == 0) {
            const uint32_t t = idx[size_t(row) * k];
            tok[row] = t;
            hist[(steps[row] % hist_cap) * rows + row] = t;
            steps[row] += 1u;   // the history slot only (greedy draws no uniform)
        }
        return;
    }
    // the valid candidates, compacted in order (the host skips empty slots)
    const float v = lane < k ? val[size_t(row) * k + lane] : -INFINITY;
    const uint32_t d = lane < k ? idx[size_t(row) * k + lane] : 0xFFFFFFFFu;
    const bool ok = d != 0xFFFFFFFFu;
    const unsigned long long m = __ballot(ok);
    const uint32_t at = uint32_t(__popcll(m & ((1ull << lane) - 1ull))), n = uint32_t(__popcll(m));
    if (ok) {
        sv[at] = v;
        si[at] = d;
    }
    __syncthreads();
    const float t = temperature > 0.0f ? temperature : 1.0f;
    const uint32_t kk = top_k ? min(top_k, n) : n;
    float maxl = -INFINITY;
    for (uint32_t i = 0; i < kk; ++i) maxl = maxl < sv[i] ? sv[i] : maxl;
    if (lane < kk) se[lane] = float(exp(double((sv[lane] - maxl) / t)));
    __syncthreads();
    if (lane != 0) return;
    uint32_t token = 0u;
    if (n > 0) {
        uint32_t nn = kk;
        double sum = 0.0;
        for (uint32_t i = 0; i < nn; ++i) sum += double(se[i]);
        if (top_p > 0.0f && top_p < 1.0f && sum > 0.0) {
            double acc = 0.0;
            const double cut = double(top_p) * sum;
            uint32_t keep = 0;
            for (; keep < nn; ++keep) {
                acc += double(se[keep]);
                if (acc >= cut) break;
            }
            nn = min(nn, keep + 1u);
            sum = 0.0;
            for (uint32_t i = 0; i < nn; ++i) sum += double(se[i]);
        }
        uint32_t o[4];
        philox4x32_10_dev(steps[row], 0u, 0u, 0u, seed, seq0 + row, o);
        const uint64_t bits = (uint64_t(o[0]) << 21) | (o[1] >> 11);
        const double u = double(bits) * (1.0 / 9007199254740992.0);
        double r = u * sum;
        token = si[nn - 1u];
        for (uint32_t i = 0; i < nn; ++i) {
            r -= double(se[i]);
            if (r <= 0.0) {
                token = si[i];
                break;
            }
        }
    }
    tok[row] = token;
    hist[(steps[row] % hist_cap) * rows + row] = token;
    steps[row] += 1u;
}

int launch_draw_rows(const float* val, const uint32_t* idx, uint32_t k, uint32_t rows, int mode,
                     float temperature, uint32_t top_k, float top_p, uint32_t seed, uint32_t seq0,
                     uint32_t* steps, uint32_t* tok, uint32_t* hist, uint32_t hist_cap, hipStream_t st) {
    if (k < 1 || k > uint32_t(kWave) || rows == 0 || hist_cap == 0)
        return set_error(XP_E_ARG, "draw rows: k=%u rows=%u hist_cap=%u", k, rows, hist_cap);
    hipLaunchKernelGGL(draw_rows_kernel, dim3(rows), dim3(kWave), 0, st, val, idx, k, mode, temperature,
                       top_k, top_p, seed, seq0, steps, tok, hist, hist_cap);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(XP_E_HIP, "draw rows: launch -> %s", hipGetErrorString(e));
    return XP_OK;
}

int launch_select_rows(float* oval, uint32_t* oidx, const float* cval, const uint32_t* cidx,
                       uint32_t ncand, uint32_t k, uint32_t rows, hipStream_t st, uint32_t* pos_inc) {
    if (k < 1 || k > kTopkMax || rows == 0 || ncand == 0 || ncand > kSelThreads * kSelPer)
        return set_error(XP_E_ARG, "select rows: k=%u rows=%u ncand=%u (<= %u)", k, rows, ncand,
                         kSelThreads * kSelPer);
    hipLaunchKernelGGL(select_rows_kernel, dim3(rows), dim3(kSelThreads), 0, st, oval, oidx, cval, cidx,
                       ncand, k, pos_inc);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(XP_E_HIP, "select rows: launch -> %s", hipGetErrorString(e));
    return XP_OK;
}

}  // namespace xp

using namespace xp;

#define XP_SC_LAUNCH(name) \
    do { \
        hipError_t e_ = hipGetLastError(); \
        if (e_ != hipSuccess) return set_error(XP_E_HIP, name ": launch -> %s", hipGetErrorString(e_)); \
        return XP_OK; \
    } while (0)

extern "C" {

int xp_apply_temperature(float* logits, float inv_temp, uint32_t n, xp_stream stream) {
    XP_REQUIRE(logits, "null pointer");
    XP_REQUIRE(n > 0, "n must be positive");
    XP_REQUIRE(std::isfinite(inv_temp), "inv_temp must be finite (route T == 0 to argmax)");
    hipLaunchKernelGGL(temperature_kernel, dim3(blocks(n, kScThreads)), dim3(kScThreads), 0,
                       as_stream(stream), logits, inv_temp, n);
    XP_SC_LAUNCH("xp_apply_temperature");
}

int xp_reduce_max_partial(float* pmax, const float* x, uint32_t n, uint32_t nparts,
                          xp_stream stream) {
    XP_REQUIRE(pmax && x, "null pointer");
    XP_REQUIRE(n > 0 && nparts > 0, "n and nparts must be positive");
    if (max_by_thread(n, nparts))
        hipLaunchKernelGGL(reduce_max_partial_thread_kernel, dim3(blocks(nparts, kScThreads)), dim3(kScThreads),
                           0, as_stream(stream), pmax, x, n, nparts);
    else
        hipLaunchKernelGGL(reduce_max_partial_kernel, dim3(blocks(nparts, kChainW)), dim3(kScThreads),
                           0, as_stream(stream), pmax, x, n, nparts);
    XP_SC_LAUNCH("xp_reduce_max_partial");
}

int xp_reduce_max_final(float* stats, const float* pmax, uint32_t nparts, xp_stream stream) {
    XP_REQUIRE(stats && pmax, "null pointer");
    XP_REQUIRE(nparts > 0, "nparts must be positive");
    hipLaunchKernelGGL(reduce_max_final_kernel, dim3(1), dim3(1024), 0, as_stream(stream), stats,
                       pmax, nparts);
    XP_SC_LAUNCH("xp_reduce_max_final");
}

int xp_softmax_exp_partial(float* out, float* psum, const float* x, const float* stats, uint32_t n,
                           uint32_t nparts, xp_stream stream) {
    XP_REQUIRE(out && psum && x && stats, "null pointer");
    XP_REQUIRE(n > 0 && nparts > 0, "n and nparts must be positive");
    if (exp_by_thread(n, nparts))
        hipLaunchKernelGGL(softmax_exp_partial_thread_kernel, dim3(blocks(nparts, kScThreads)), dim3(kScThreads),
                           0, as_stream(stream), out, psum, x, stats, n, nparts);
    else
        hipLaunchKernelGGL(softmax_exp_partial_kernel, dim3(blocks(nparts, kChainW)), dim3(kScThreads),
                           0, as_stream(stream), out, psum, x, stats, n, nparts);
    XP_SC_LAUNCH("xp_softmax_exp_partial");
}

int xp_reduce_sum_partial(float* out, const float* in, uint32_t n, uint32_t nparts,
                          xp_stream stream) {
    XP_REQUIRE(out && in, "null pointer");
    XP_REQUIRE(n > 0 && nparts > 0, "n and nparts must be positive");
    hipLaunchKernelGGL(reduce_sum_partial_kernel, dim3(blocks(nparts, kScThreads)), dim3(kScThreads),
                       0, as_stream(stream), out, in, n, nparts);
    XP_SC_LAUNCH("xp_reduce_sum_partial");
}

int xp_reduce_sum_final(float* stats, const float* psum, uint32_t nparts, xp_stream stream) {
    XP_REQUIRE(stats && psum, "null pointer");
    XP_REQUIRE(nparts > 0, "nparts must be positive");
    hipLaunchKernelGGL(reduce_sum_final_kernel, dim3(1), dim3(kScThreads), 0, as_stream(stream), stats, psum,
                       nparts);
    XP_SC_LAUNCH("xp_reduce_sum_final");
}

int xp_softmax_normalize(float* out, const float* stats, uint32_t n, xp_stream stream) {
    XP_REQUIRE(out && stats, "null pointer");
    XP_REQUIRE(n > 0, "n must be positive");
    hipLaunchKernelGGL(softmax_normalize_kernel, dim3(blocks(n, kScThreads)), dim3(kScThreads), 0,
                       as_stream(stream), out, stats, n);
    XP_SC_LAUNCH("xp_softmax_normalize");
}

int xp_topk_partial(float* cval, uint32_t* cidx, const float* x, uint32_t n, uint32_t nparts,
                    uint32_t k, xp_stream stream) {
    XP_REQUIRE(cval && cidx && x, "null pointer");
    XP_REQUIRE(n > 0 && nparts > 0, "n and nparts must be positive");
    XP_REQUIRE(k >= 1 && k <= kTopkMax, "k=%u must be in [1, %u]", k, kTopkMax);
    if (topk_by_wave(n, nparts, k))
        hipLaunchKernelGGL(topk_partial_wave_kernel, dim3(nparts), dim3(kWave), 0, as_stream(stream), cval, cidx, x,
                           n, nparts, k);
    else
        hipLaunchKernelGGL(topk_partial_kernel, dim3(blocks(nparts, kTopkThreads)), dim3(kTopkThreads), 0,
                           as_stream(stream), cval, cidx, x, n, nparts, k);
    XP_SC_LAUNCH("xp_topk_partial");
}

int xp_topk_rank_select(float* oval, uint32_t* oidx, const float* cval, const uint32_t* cidx,
                        uint32_t ncand, uint32_t k, xp_stream stream) {
    XP_REQUIRE(oval && oidx && cval && cidx, "null pointer");
    XP_REQUIRE(ncand > 0 && k > 0, "ncand and k must be positive");
    // the scan counts every candidate against all, half a us for each 64 of
    // them; the search has its 5.2 to 6.8 us from the first (64 candidates 4.1
    // against 5.2-5.9, 128 5.5 against 5.4-6.7, 192 7.4 against 5.2-7.0)
    if (ncand > 128u && k <= kTopkMax)
        hipLaunchKernelGGL(topk_rank_wave_kernel, dim3(1), dim3(kWave * std::min(16u, blocks(ncand, 1024u))), 0,
                           as_stream(stream), oval, oidx, cval, cidx, ncand, k);
    else
        hipLaunchKernelGGL(topk_rank_select_kernel, dim3(blocks(ncand, kScThreads)), dim3(kScThreads), 0,
                           as_stream(stream), oval, oidx, cval, cidx, ncand, k);
    XP_SC_LAUNCH("xp_topk_rank_select");
}

int xp_topk_mask(float* logits, const float* topk_val, uint32_t k, uint32_t n, xp_stream stream) {
    XP_REQUIRE(logits && topk_val, "null pointer");
    XP_REQUIRE(n > 0 && k > 0, "n and k must be positive");
    hipLaunchKernelGGL(topk_mask_kernel, dim3(blocks(n, kScThreads)), dim3(kScThreads), 0,
                       as_stream(stream), logits, topk_val, k, n);
    XP_SC_LAUNCH("xp_topk_mask");
}

int xp_topp_cutoff(float* w, uint32_t k, float p, xp_stream stream) {
    XP_REQUIRE(w, "null pointer");
    XP_REQUIRE(k > 0, "k must be positive");
    hipLaunchKernelGGL(topp_cutoff_kernel, dim3(1), dim3(64), 0, as_stream(stream), w, k, p);
    XP_SC_LAUNCH("xp_topp_cutoff");
}

int xp_multinomial_sample(float* out, uint32_t* idx_out, const float* w, const uint32_t* idx,
                          uint32_t k, float u, xp_stream stream) {
    XP_REQUIRE(out && idx_out && w && idx, "null pointer");
    XP_REQUIRE(k > 0, "k must be positive");
    hipLaunchKernelGGL(multinomial_sample_kernel, dim3(1), dim3(64), 0, as_stream(stream), out, idx_out,
                       w, idx, k, u);
    XP_SC_LAUNCH("xp_multinomial_sample");
}

int xp_multinomial_strided(float* out, uint32_t* idx_out, const float* w, const float* psum,
                           const float* stats, uint32_t n, uint32_t nparts, float u,
                           xp_stream stream) {
    XP_REQUIRE(out && idx_out && w && psum && stats, "null pointer");
    XP_REQUIRE(n > 0 && nparts > 0 && nparts <= n, "need 0 < nparts <= n");
    hipLaunchKernelGGL(multinomial_strided_kernel, dim3(1), dim3(kScThreads), 0, as_stream(stream), out,
                       idx_out, w, psum, stats, n, nparts, u);
    XP_SC_LAUNCH("xp_multinomial_strided");
}

}  // extern "C"
