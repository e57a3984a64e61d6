// kernels_topk.hip -- per-query k smallest cRMSD values of a score row, ties
// to the lower library index, sorted by (value, index).
//
// Rows of up to kRowMax values (topk_row_kernel): one work-group holds the row
// in registers, bisects the key space down to a few hundred candidates and
// sorts those.  Longer rows take two stages:
//  1. topk_chunk_kernel: one work-group per (chunk of a row, query).  The
//     chunk's k-th smallest key is found by a three-pass radix select (11 + 11
//     + 10 bits; non-negative floats order like their bit patterns) with
//     per-wave LDS histograms and a block-wide scan over the bins; the keys
//     below it and, in index order, enough keys equal to it are written out as
//     (key << 32 | index) candidates.
//  2. topk_merge_kernel: one work-group per query sorts the row's candidates
//     (at most kMergeMax, chunk sizes are chosen so) with a bitonic sort in
//     LDS and writes the first k.
// The k smallest (value, index) pairs of a row are among the union of every
// chunk's k smallest, so the result is exact.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace bs {
namespace {

constexpr int kTopkMax = 1024;
constexpr int kMergeMax = 8192;
constexpr int kChunkThreads = 256;
constexpr int kChunkWaves = kChunkThreads / 64;
constexpr int kMinChunk = 4096;
constexpr int kCachedKeys = kMinChunk / kChunkThreads;  // keys per thread kept in registers

__device__ inline uint32_t key_of(float v)
{
    uint32_t u = __float_as_uint(v);
    if (v != v) return 0x7FC00000u;  // NaN sorts after every number
    if (u & 0x80000000u) return 0u;  // -0 and negatives (never produced) first
    return u;
}

// Exclusive scan of one value per thread over the block (256 threads);
// returns the thread's prefix, *total gets the block sum.
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_wave, uint32_t* total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[w] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < kChunkWaves; ++k) {
        const uint32_t t = s_wave[k];
        if (k < w) before += t;
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + x - v;
}

__global__ __launch_bounds__(kChunkThreads) void topk_chunk_kernel(const float* __restrict__ scores, int n,
                                                                   int k, int chunk,
                                                                   unsigned long long* __restrict__ cand)
{
    __shared__ uint32_t hist[kChunkWaves][2048];
    __shared__ uint32_t s_wave[kChunkWaves];
    __shared__ uint32_t s_bin, s_need, s_cnt;
    __shared__ uint32_t eq_cnt[kChunkWaves * 129];
    const int q = blockIdx.y, c = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int base = c * chunk;
    const int len = min(chunk, n - base);
    const int kc = min(k, len);
    const float* row = scores + (int64_t)q * n + base;
    unsigned long long* out = cand + ((int64_t)q * gridDim.x + c) * k;

    // the thread's first kCachedKeys keys (elements tid, tid + 256, ...) are
    // read once and kept in registers for every pass; a longer chunk reads
    // the rest from memory each time
    uint32_t keys[kCachedKeys];
#pragma unroll
    for (int j = 0; j < kCachedKeys; ++j) {
        const int e = j * kChunkThreads + tid;
        keys[j] = e < len ? key_of(row[e]) : 0xFFFFFFFFu;
    }
    auto key_at = [&](int j, int e) { return j < kCachedKeys ? keys[j] : key_of(row[e]); };
    const int iters = (len + kChunkThreads - 1) / kChunkThreads;  // <= 128 (chunk <= 32768)

    uint32_t prefix = 0, pmask = 0, need = (uint32_t)kc;
    for (int pass = 0; pass < 3; ++pass) {
        const int shift = pass == 0 ? 21 : (pass == 1 ? 10 : 0);
        const int nb = pass < 2 ? 2048 : 1024;
        for (int b = tid; b < kChunkWaves * 2048; b += kChunkThreads) (&hist[0][0])[b] = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kCachedKeys; ++j) {
            const uint32_t key = keys[j];
            if (j * kChunkThreads + tid < len && (key & pmask) == prefix)
                atomicAdd(&hist[wv][(key >> shift) & (nb - 1)], 1u);
        }
        for (int e = kCachedKeys * kChunkThreads + tid; e < len; e += kChunkThreads) {
            const uint32_t key = key_of(row[e]);
            if ((key & pmask) == prefix) atomicAdd(&hist[wv][(key >> shift) & (nb - 1)], 1u);
        }
        __syncthreads();
        // thread t owns bins [8t, 8t + 8): the bin where the running count reaches `need`
        const int per = nb / kChunkThreads;
        uint32_t own[8], sum = 0;
        for (int i = 0; i < per; ++i) {
            const int b = tid * per + i;
            own[i] = hist[0][b] + hist[1][b] + hist[2][b] + hist[3][b];
            sum += own[i];
        }
        uint32_t total;
        const uint32_t before = block_exclusive_scan(sum, s_wave, &total);
        if (before < need && before + sum >= need) {
            uint32_t cum = before;
            int i = 0;
            for (; i < per - 1; ++i) {
                if (cum + own[i] >= need) break;
                cum += own[i];
            }
            s_bin = (uint32_t)(tid * per + i);
            s_need = need - cum;
        }
        __syncthreads();
        prefix |= s_bin << shift;
        pmask |= (uint32_t)(nb - 1) << shift;
        need = s_need;
        __syncthreads();
    }
    const uint32_t T = prefix;  // the kc-th smallest key; `need` copies of it are taken
    // rank the keys equal to T in index order: counts per (iteration, wave), one scan
    for (int j = 0; j < iters; ++j) {
        const int e = j * kChunkThreads + tid;
        const bool eq = e < len && key_at(j, e) == T;
        const uint64_t m = __ballot(eq);
        if (lane == 0) eq_cnt[j * kChunkWaves + wv] = (uint32_t)__popcll(m);
    }
    if (tid == 0) s_cnt = 0;
    __syncthreads();
    {
        // exclusive prefix over the (iteration, wave) counts, two entries per thread
        const int n_e = iters * kChunkWaves, i0 = 2 * tid;
        const uint32_t a = i0 < n_e ? eq_cnt[i0] : 0u, b = i0 + 1 < n_e ? eq_cnt[i0 + 1] : 0u;
        uint32_t total;
        const uint32_t before = block_exclusive_scan(a + b, s_wave, &total);
        if (i0 < n_e) eq_cnt[i0] = before;
        if (i0 + 1 < n_e) eq_cnt[i0 + 1] = before + a;
    }
    __syncthreads();
    for (int j = 0; j < iters; ++j) {
        const int e = j * kChunkThreads + tid;
        const uint32_t key = e < len ? key_at(j, e) : 0xFFFFFFFFu;
        const bool lt = e < len && key < T;
        const bool eq = e < len && key == T;
        const uint64_t m = __ballot(eq);
        const uint32_t below = (uint32_t)__popcll(m & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
        const bool take = lt || (eq && eq_cnt[j * kChunkWaves + wv] + below < need);
        if (take) {
            const uint32_t pos = atomicAdd(&s_cnt, 1u);
            if (pos < (uint32_t)kc) out[pos] = ((unsigned long long)key << 32) | (uint32_t)(base + e);
        }
    }
    for (int v = kc + tid; v < k; v += kChunkThreads) out[v] = ~0ull;  // short last chunk
}

// Sorts the P (a power of two) values at s, by 1024 threads; starts and ends at
// a barrier.
__device__ inline void bitonic_sort(unsigned long long* s, int P)
{
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int v = threadIdx.x; v < P; v += 1024) {
                const int w = v ^ stride;
                if (w > v) {
                    const bool up = (v & size) == 0;
                    const unsigned long long x = s[v], y = s[w];
                    if ((x > y) == up) {
                        s[v] = y;
                        s[w] = x;
                    }
                }
            }
            __syncthreads();
        }
}

__global__ __launch_bounds__(1024) void topk_merge_kernel(const unsigned long long* __restrict__ cand, int m,
                                                          int k, uint32_t* __restrict__ out_idx,
                                                          float* __restrict__ out_val, uint64_t* t_end)
{
    __shared__ unsigned long long s[kMergeMax];
    const int q = blockIdx.x, tid = threadIdx.x;
    const unsigned long long* in = cand + (int64_t)q * m;
    int P = 1;
    while (P < m) P <<= 1;
    for (int v = tid; v < P; v += 1024) s[v] = v < m ? in[v] : ~0ull;
    __syncthreads();
    bitonic_sort(s, P);
    for (int v = tid; v < k; v += 1024) {
        const unsigned long long c = s[v];
        out_idx[(int64_t)q * k + v] = (uint32_t)(c & 0xFFFFFFFFu);
        out_val[(int64_t)q * k + v] = __uint_as_float((uint32_t)(c >> 32));
    }
    stamp_end(t_end);
}

// One row in the registers of one work-group, KPT keys per thread (element
// j * 1024 + thread).  Non-negative floats order like their bit patterns, so a
// threshold with at least k and at most kRowCand / 2, or 256, keys at or below
// it is found by bisecting the integers between the row's smallest and largest
// key, counting first the threads' smallest keys, then all.  Where the
// bisection ends at one key (more equal keys than that), it is the k-th
// smallest, and of its copies the first in index order are taken.  The
// candidates are sorted by (key, index), each by counting the smaller ones
// (up to 1024) or all by a bitonic sort, and the first k written.
// Bound by latency: 25,000 values, k 100, 32 rows: 13.4 us, where a radix
// select of 4096-value chunks and a bitonic merge took 18.3 + 17.2 (bisecting
// over all keys from the start: 17.5).
constexpr int kRowThreads = 1024;
constexpr int kRowWaves = kRowThreads / 64;
constexpr int kRowKeys = 32;  // at most, per thread
constexpr int kRowMax = kRowThreads * kRowKeys;
constexpr int kRowCand = 2048;

template <int KPT>
__global__ __launch_bounds__(kRowThreads) void topk_row_kernel(const float* __restrict__ scores, int n, int k,
                                                               uint32_t* __restrict__ out_idx,
                                                               float* __restrict__ out_val, uint64_t* t_end)
{
    __shared__ __align__(16) unsigned long long cand[kRowCand];
    __shared__ uint32_t rank[kRowThreads];
    __shared__ uint32_t s_lo[kRowWaves], s_hi[kRowWaves], s_cnt[2][kRowWaves], s_eq[kRowKeys * kRowWaves], s_n;
    const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const float* row = scores + (int64_t)q * n;
    uint32_t keys[KPT];
    uint32_t mn = 0xFFFFFFFFu, mx = 0u;
    {
        float v[KPT];  // clamped addresses: every load in flight at once
#pragma unroll
        for (int j = 0; j < KPT; ++j) v[j] = row[min(j * kRowThreads + tid, n - 1)];
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
            const bool in = j * kRowThreads + tid < n;
            const uint32_t key = key_of(v[j]);
            keys[j] = in ? key : 0xFFFFFFFFu;
            mn = min(mn, keys[j]);
            mx = max(mx, in ? key : 0u);
        }
    }
    const uint32_t own_min = mn;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, o));
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
    }
    if (lane == 0) {
        s_lo[wv] = mn;
        s_hi[wv] = mx;
    }
    if (tid == 0) s_n = 0;
    rank[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) {
        mn = min(mn, s_lo[w]);
        mx = max(mx, s_hi[w]);
    }
    // fewer than k keys are <= lo (as integers; below the smallest key), c_hi >= k are <= hi
    const uint32_t cap = k <= 128 ? 256u : (k <= 512 ? 1024u : (uint32_t)kRowCand);
    int64_t lo = (int64_t)mn - 1, hi = (int64_t)mx;
    uint32_t c_lo = 0, c_hi = (uint32_t)n;
    int buf = 0;
    auto block_sum = [&](uint32_t c) {
        if (lane == 0) s_cnt[buf][wv] = c;
        __syncthreads();
        c = 0;
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w) c += s_cnt[buf][w];
        buf ^= 1;  // the next sum's words are not those some wave may still read
        return c;
    };
    auto count = [&](uint32_t t) {
        uint32_t c = 0;
#pragma unroll
        for (int j = 0; j < KPT; ++j) c += (uint32_t)__popcll(__ballot(keys[j] <= t));
        return block_sum(c);
    };
    // first over the threads' smallest keys, one compare each: k of those at
    // or below a threshold are k keys, and for a row in no special order few
    // more keys than that are
    if (c_hi > cap && k <= kRowThreads / 2) {
        int64_t l = lo;
        uint32_t c = kRowThreads;
        while (c > cap / 2 + (uint32_t)k / 2 && hi - l > 1) {
            const int64_t mid = l + (hi - l) / 2;
            const uint32_t m = block_sum((uint32_t)__popcll(__ballot(own_min <= (uint32_t)mid)));
            if (m >= (uint32_t)k) {
                hi = mid;
                c = m;
            } else {
                l = mid;
            }
        }
        c_hi = count((uint32_t)hi);
    }
    while (c_hi > cap && hi - lo > 1) {
        const int64_t mid = lo + (hi - lo) / 2;
        const uint32_t c = count((uint32_t)mid);
        if (c >= (uint32_t)k) {
            hi = mid;
            c_hi = c;
        } else {
            lo = mid;
            c_lo = c;
        }
    }
    const bool ties = c_hi > cap;  // uniform: hi is the k-th smallest key, k - c_lo copies of it are taken
    const uint64_t lower = (1ull << lane) - 1ull;
    if (!ties || lo >= 0) {
        // the keys at or below hi, or below it
        const uint32_t t = (uint32_t)(ties ? lo : hi);
        uint32_t mine = 0;
#pragma unroll
        for (int j = 0; j < KPT; ++j) mine += keys[j] <= t ? 1u : 0u;
        if (mine) {
            uint32_t pos = atomicAdd(&s_n, mine);
#pragma unroll
            for (int j = 0; j < KPT; ++j)
                if (keys[j] <= t) cand[pos++] = ((unsigned long long)keys[j] << 32) | (uint32_t)(j * kRowThreads + tid);
        }
    }
    if (ties) {
        // copies of the k-th key in index order: counts per (iteration, wave), their prefix sums, then places
        const int iters = (n + kRowThreads - 1) / kRowThreads;
        const uint32_t T = (uint32_t)hi, need = (uint32_t)k - c_lo;
        auto equal = [&](int j) {
            const int e = j * kRowThreads + tid;
            return e < n && key_of(row[min(e, n - 1)]) == T;
        };
#pragma unroll 1
        for (int j = 0; j < iters; ++j) {
            const uint32_t m = (uint32_t)__popcll(__ballot(equal(j)));
            if (lane == 0) s_eq[j * kRowWaves + wv] = m;
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t sum = 0;
            for (int i = 0; i < iters * kRowWaves; ++i) {
                const uint32_t m = s_eq[i];
                s_eq[i] = sum;
                sum += m;
            }
            s_n = (uint32_t)k;
        }
        __syncthreads();
#pragma unroll 1
        for (int j = 0; j < iters; ++j) {
            const bool eq = equal(j);
            const uint32_t at = s_eq[j * kRowWaves + wv] + (uint32_t)__popcll(__ballot(eq) & lower);
            if (eq && at < need)
                cand[c_lo + at] = ((unsigned long long)T << 32) | (uint32_t)(j * kRowThreads + tid);
        }
    }
    __syncthreads();
    const int m = (int)s_n;
    int P = 64;
    while (P < m) P <<= 1;
    for (int v = m + tid; v < P; v += kRowThreads) cand[v] = ~0ull;
    __syncthreads();
    uint32_t* oi = out_idx + (int64_t)q * k;
    float* ov = out_val + (int64_t)q * k;
    if (P <= kRowThreads) {
        // 1024 / P threads per candidate, each counting the smaller ones among its share
        const int i = tid & (P - 1), share = P * P / kRowThreads;  // of P >= 64 candidates: a multiple of 4
        const unsigned long long own = cand[i];
        const ulonglong2* c2 = reinterpret_cast<const ulonglong2*>(cand + tid / P * share);
        uint32_t less = 0;
#pragma unroll 8
        for (int v = 0; v < share / 2; ++v) {
            const ulonglong2 c = c2[v];
            less += (c.x < own ? 1u : 0u) + (c.y < own ? 1u : 0u);
        }
        if (less) atomicAdd(&rank[i], less);
        __syncthreads();
        if (tid < m && rank[tid] < (uint32_t)k) cand[rank[tid]] = own;
        __syncthreads();
    } else {
        bitonic_sort(cand, P);
    }
    // in order: the results may be in host memory, where single words are slow
    for (int v = tid; v < k; v += kRowThreads) {
        oi[v] = (uint32_t)(cand[v] & 0xFFFFFFFFu);
        ov[v] = __uint_as_float((uint32_t)(cand[v] >> 32));
    }
    stamp_end(t_end);
}

// Chunk length: at least kMinChunk, a multiple of 256, and few enough chunks
// that a row's candidates (chunks x k) fit the merge.
int topk_chunk_len(int n_lib, int k)
{
    const int max_chunks = std::max(1, kMergeMax / std::max(k, 1));
    int c = (n_lib + max_chunks - 1) / max_chunks;
    c = std::max(c, kMinChunk);
    return (c + kChunkThreads - 1) / kChunkThreads * kChunkThreads;
}

}  // namespace

size_t topk_scratch_bytes(int n_q, int n_lib, int k)
{
    if (n_q <= 0 || k <= 0) return 0;
    const int chunk = topk_chunk_len(n_lib, k);
    const int n_chunks = (n_lib + chunk - 1) / chunk;
    return (size_t)n_q * n_chunks * k * 8;
}

bool topk_supported(int n_lib, int k)
{
    if (k <= 0 || k > kTopkMax || k > n_lib) return false;
    const int chunk = topk_chunk_len(n_lib, k);
    const int n_chunks = (n_lib + chunk - 1) / chunk;
    return chunk <= 128 * kChunkThreads && n_chunks * k <= kMergeMax;
}

void launch_topk(const float* scores, int n_q, int n_lib, int k, uint32_t* idx, float* val, void* scratch,
                 hipStream_t s, uint64_t* t_end)
{
    if (n_q <= 0) return;
    if (k <= 0 || k > kTopkMax || k > n_lib) fail(BS_ERR_INVALID_ARGUMENT, "top-k: k = %d outside [1, min(%d, %d)]",
                                                  k, kTopkMax, n_lib);
    if (!topk_supported(n_lib, k))
        fail(BS_ERR_UNSUPPORTED, "top-k: %d library members with k = %d exceed the selection's range", n_lib, k);
    if (n_lib <= kRowMax) {
        if (n_lib <= 8 * kRowThreads)
            topk_row_kernel<8><<<n_q, kRowThreads, 0, s>>>(scores, n_lib, k, idx, val, t_end);
        else if (n_lib <= 16 * kRowThreads)
            topk_row_kernel<16><<<n_q, kRowThreads, 0, s>>>(scores, n_lib, k, idx, val, t_end);
        else
            topk_row_kernel<kRowKeys><<<n_q, kRowThreads, 0, s>>>(scores, n_lib, k, idx, val, t_end);
        return;
    }
    const int chunk = topk_chunk_len(n_lib, k);
    const int n_chunks = (n_lib + chunk - 1) / chunk;
    auto* cand = static_cast<unsigned long long*>(scratch);
    topk_chunk_kernel<<<dim3(n_chunks, n_q), kChunkThreads, 0, s>>>(scores, n_lib, k, chunk, cand);
    topk_merge_kernel<<<n_q, 1024, 0, s>>>(cand, n_chunks * k, k, idx, val, t_end);
}

}  // namespace bs
