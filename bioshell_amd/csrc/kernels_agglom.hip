// kernels_agglom.hip -- the whole agglomeration loop of hierarchical
// clustering in one cooperative launch, for up to 16,384 elements (labels of 14
// bits; the caches then fit the LDS of 224 CUs).
//
// The loop is the reference's (clustering_matrix.rs; the rules of the merge,
// of the move and of ties are listed in kernels_cluster.hip), and its merge
// sequence is the same bit for bit.  What differs is how much is read per
// merge:
//  - Rows stay where they are.  An element's place in the matrix is its slot;
//    the reference's moving index is a label, kept per slot, so the move of
//    the last cluster to index j changes one label instead of a row and a
//    column.
//  - Every row caches its smallest entry per block of 64 columns (in LDS) and
//    over the row.  A merge of slots I and J changes a row's entries at I, J
//    and, by its new label, at L: the blocks of I and J are scanned again if
//    their cached minimum was there, and the row's minimum is taken from the
//    blocks only if it was.  With average linkage about one block scan per row
//    and merge replaces a scan of the whole row, where the stepwise kernels read
//    67 MB a merge at 10,000 elements.
//  - A row belongs to one wave, which alone reads and writes it, through
//    ordinary cached accesses; only the merged row is written by its whole
//    work-group, a step's barrier before its wave reads it again.  What a merge
//    needs from other work-groups goes through small exchange buffers with
//    agent-scope accesses: every work-group's best candidate (slots) and the
//    merged row's new entries (newrow), each element's from the owner of its
//    row.  Storing a candidate is also the arrival at
//    the step's barrier: everyone polls the slots until none is empty.  The
//    buffers rotate by three: a work-group that has seen every candidate of
//    step s knows that all have read those of step s - 1.
//  - The merged row itself joins the matrix a step later, while the next
//    candidates are on their way.  Until then its owner reads its entries from
//    newrow; the other pairs of that row are covered by their other element's
//    row, whose caches have the new entry at once.
//
// Bound: latency.  Of 4.2 us per merge at 300 elements (12 work-groups) about
// 1.3 us are the exchange and the rest the dependent steps of one wave, of 7.1
// us at 10,000 (224 work-groups) about 3.4; memory traffic is below 0.5 TB/s.
// Against two launches per merge: 300 elements 3.2 -> 1.3 ms, 2000 20 -> 10.5
// ms, 10,000 193 -> 71 ms, 16,300 745 -> 240 ms (average linkage).  Measured and not kept: one
// work-group without the exchange (as fast up to 180 elements, slower above),
// the matrix in LDS (3 % at 300 to 2000 elements), 8 waves per work-group (a
// step is bound by the instructions of its waves).
#include <algorithm>

#include "cluster_rule.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace bs {
namespace {

constexpr unsigned kDead = 0xFFFFu;
constexpr uint64_t kNone = ~0ull;       // no candidate
constexpr uint64_t kAgain = ~0ull - 1;  // a row minimum to be taken from the block minima
constexpr int kMaxElements = 16384;     // labels take 14 bits of a published key
constexpr int kLdsBytes = 160 * 1024;
constexpr int kWaves = 4;               // per work-group
constexpr int kRowsWanted = 24;         // rows per work-group while the device has CUs for it
constexpr int kWaveItems = 2 * 64;      // blocks a wave may have to scan again in a step
constexpr int kUnroll = 4;              // block scans in flight per quarter wave
constexpr int kCopy = 8;                // runs of a merged row in flight per quarter wave
constexpr float kFltMax = 3.402823466e+38f;

// A row's candidate: value (order-preserving bits, -0 as +0), the partner's
// current index, and in the lowest bit the value's sign (of a zero).
__device__ inline uint64_t row_key(float v, unsigned label)
{
    const uint64_t k =
        ((uint64_t)fkey(__float_as_uint(v + 0.0f)) << 32) | (label << 1) | (__float_as_uint(v) >> 31);
    return v < kFltMax ? k : kNone;  // NaN and values from f32::MAX on are never taken
}
__device__ inline uint64_t lesser(uint64_t a, uint64_t b) { return b < a ? b : a; }
__device__ inline unsigned key_label(uint64_t k) { return (unsigned)k >> 1; }

// The smallest of the 16 lanes of a row, in each of them.
__device__ inline unsigned min16_u32(unsigned v)
{
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, true));  // row_ror:8
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, true));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xF, 0xF, true));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xF, 0xF, true));
    return v;
}
__device__ inline uint64_t min16_u64(uint64_t k)
{
    const unsigned hi = min16_u32((unsigned)(k >> 32));
    const unsigned lo = min16_u32((unsigned)(k >> 32) == hi ? (unsigned)k : ~0u);
    return ((uint64_t)hi << 32) | lo;
}
// The same over the 64 lanes (uniform).
__device__ inline unsigned min64_u32(unsigned v)
{
    v = min(v, dpp_u32<0x111, 0xF>(v, ~0u));
    v = min(v, dpp_u32<0x112, 0xF>(v, ~0u));
    v = min(v, dpp_u32<0x114, 0xF>(v, ~0u));
    v = min(v, dpp_u32<0x118, 0xF>(v, ~0u));
    v = min(v, dpp_u32<0x142, 0xA>(v, ~0u));
    v = min(v, dpp_u32<0x143, 0xC>(v, ~0u));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ inline uint64_t min64_u64(uint64_t k)
{
    const unsigned hi = min64_u32((unsigned)(k >> 32));
    const unsigned lo = min64_u32((unsigned)(k >> 32) == hi ? (unsigned)k : ~0u);
    return ((uint64_t)hi << 32) | lo;
}

// Smallest key of one block of a row, by 16 lanes: each lane's smallest value
// and, among the columns that hold the row's smallest, the smallest label.
// x holds the lane's values of columns c .. c + 3 (absent ones as +inf).
struct QuadMin {
    float v;
    unsigned l;  // label << 1 | sign
};
__device__ inline void quad_take(QuadMin& m, const float (&x)[4], const uint16_t* label, int c)
{
    const ushort4 l4 = *reinterpret_cast<const ushort4*>(label + c);
    const unsigned ls[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const unsigned l = (ls[u] << 1) | (__float_as_uint(x[u]) >> 31);
        const bool better = (x[u] < m.v) | ((x[u] == m.v) & (l < m.l));
        m.v = better ? x[u] : m.v;
        m.l = better ? l : m.l;
    }
}
__device__ inline uint64_t quad_key16(const QuadMin& m)
{
    const unsigned k = m.v < kFltMax ? fkey(__float_as_uint(m.v + 0.0f)) : ~0u;
    const unsigned hi = min16_u32(k);
    const unsigned lo = min16_u32(k == hi ? m.l : ~0u);
    return hi == ~0u ? kNone : ((uint64_t)hi << 32) | lo;
}

template <class V>
__device__ inline void agent_store(V* p, V v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class V>
__device__ inline V agent_load(const V* p)
{
    return __hip_atomic_load(const_cast<V*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <bool WIDE, int RULE>
__global__ __launch_bounds__(64 * kWaves) void agglom_kernel(AgglomArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int W = kWaves, T = 64 * W;
    const int64_t ld = a.ld;
    const int n = a.n, R = a.rows, NB = a.n_blocks, sh = WIDE ? a.block_shift : 6, G = gridDim.x, g = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, sub = lane & 15, quarter = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int cap = NB << sh;  // columns, padded to whole blocks
    float* const D = a.D + g * ld;  // the work-group's rows: every G-th
    const int64_t step = G * ld;
    uint64_t* bm = reinterpret_cast<uint64_t*>(smem);
    uint64_t* rowbest = bm + (size_t)R * NB;
    uint64_t* wbest = rowbest + R;  // the waves' minima of the candidates read
    uint64_t* gbest = wbest + W;    // and of their own rows
    uint16_t* label = reinterpret_cast<uint16_t*>(gbest + W);
    uint16_t* slot = label + cap;
    unsigned* sizes = reinterpret_cast<unsigned*>(slot + ((n + 3) & ~3));
    unsigned* items = sizes + ((n + 3) & ~3) + w * kWaveItems;
    unsigned* ctl = sizes + ((n + 3) & ~3) + W * kWaveItems;
    const int r = lane * W + w, p = r * G + g;  // this lane's row, and its slot
    const bool own = r < R && p < n;
    float* const row = D + (own ? r : 0) * step;
    const float kInf = __builtin_inff();

    // minimum over row rr's cached block minima, by 16 lanes
    auto row_min16 = [&](int rr, bool on) -> uint64_t {
        uint64_t k = kNone;
        if (on)
            for (int b = sub; b < NB; b += 16) k = lesser(k, bm[rr * NB + b]);
        return min16_u64(k);
    };
    auto first_min = [&](const uint64_t* v) -> uint64_t {  // of W waves' minima
        uint64_t k = v[0];
#pragma unroll
        for (int u = 1; u < W; ++u) k = lesser(k, v[u]);
        return k;
    };

    for (int q = t; q < n; q += T) {
        sizes[q] = 1u;
        slot[q] = (uint16_t)q;
    }
    for (int q = t; q < cap; q += T) label[q] = q < n ? (uint16_t)q : (uint16_t)kDead;
    if (t == 0) ctl[0] = 0u;
    __syncthreads();
    for (int base = w * 4; base < R * NB; base += W * 4) {
        const int it = base + quarter;
        QuadMin m = {kFltMax, ~0u};
        if (it < R * NB) {
            const int rr = it / NB, b = it - rr * NB, pp = rr * G + g;
            if (pp < n)
                for (int c = (b << sh) + sub * 4; c < min((b + 1) << sh, (int)ld); c += 64) {
                    const float4 v = *reinterpret_cast<const float4*>(D + rr * step + c);
                    const float x[4] = {v.x, v.y, v.z, v.w};
                    quad_take(m, x, label, c);
                }
        }
        const uint64_t k = quad_key16(m);
        if (sub == 15 && it < R * NB) bm[it] = k;
    }
    __syncthreads();
    for (int base = w * 4; base < R; base += W * 4) {
        const uint64_t k = row_min16(base + quarter, base + quarter < R);
        if (sub == 15 && base + quarter < R) rowbest[base + quarter] = k;
    }
    __syncthreads();

    // the row's candidate as a published key: value, larger index, smaller index
    auto published = [&](uint64_t k, unsigned lp) -> uint64_t {
        const unsigned lq = key_label(k);
        const unsigned lo = (max(lp, lq) << 18) | (min(lp, lq) << 4) | ((unsigned)k & 1u);
        return k == kNone ? kNone : (k & 0xFFFFFFFF00000000ull) | lo;
    };
    {
        const uint64_t k = min64_u64(own ? published(rowbest[r], (unsigned)p) : kNone);
        if (lane == 0) gbest[w] = k;
        __syncthreads();
    }
    if (w == 0) {
        const uint64_t k = first_min(gbest);
        if (lane == 0) agent_store(a.slots + g, k);
    }
    int pend = -1;  // the slot merged in the step before, when its row is one of this work-group's

    for (int s = 0; s < n - 1; ++s) {
        const int order = n - s;
        {
            uint64_t k = kNone;
            if (t < G) {
                const uint64_t* q = a.slots + (size_t)(s % 3) * G + t;
                const uint64_t t0 = wall_clock64();
                int spin = 0;
                while ((k = agent_load(q)) == 0ull || a.max_wait == 0) {  // 0: gives up at once
                    if (a.max_wait == 0 || ((++spin & 255) == 0 && wall_clock64() - t0 > a.max_wait)) {
                        ctl[0] = 1u;
                        break;
                    }
                }
            }
            k = min64_u64(k);
            if (lane == 0) wbest[w] = k;
        }
        __syncthreads();
        if (ctl[0]) {  // some work-group never came: every one leaves by the same limit
            if (t == 0) agent_store(a.status, 1u);
            return;
        }
        const uint64_t best = first_min(wbest);
        // uniform: the decision and what follows from it in scalar registers
        const unsigned blo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)best);
        const unsigned bhi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(best >> 32));
        const bool none = bhi == ~0u;  // no value below f32::MAX: the reference keeps (0, 0)
        const unsigned i = none ? 0u : (blo >> 4) & 0x3FFFu;
        const unsigned j = none ? 0u : blo >> 18;
        const float dij = none ? 0.0f : ((blo & 1u) && bhi == 0x80000000u ? -0.0f : __uint_as_float(fkey_inverse(bhi)));
        const unsigned last = (unsigned)order - 1u;
        const bool moved = j < last;
        const int I = __builtin_amdgcn_readfirstlane((int)slot[i]);
        const int J = __builtin_amdgcn_readfirstlane((int)slot[j]);
        const int Ls = __builtin_amdgcn_readfirstlane((int)slot[last]);
        const int L = moved ? Ls : -1;
        const unsigned si = (unsigned)__builtin_amdgcn_readfirstlane((int)sizes[i]);
        const unsigned sj = (unsigned)__builtin_amdgcn_readfirstlane((int)sizes[j]);
        const int bI = I >> sh, bJ = J >> sh, bL = moved ? L >> sh : -1;
        const float* prev = a.newrow + (size_t)((s + 2) % 3) * ld;
        float* next = a.newrow + (size_t)(s % 3) * ld;
        auto prev_pair = [&](int q) {  // q even
            return __builtin_bit_cast(float2, agent_load(reinterpret_cast<const uint64_t*>(prev + q)));
        };

        // this lane's row: its old entries at I, J and L, in flight while the
        // blocks whose cached minimum was one of them are scanned again
        const unsigned lp = own ? label[p] : kDead;
        const bool live = (lp != kDead) & (p != I) & (p != J), fresh = live & (p == pend), scan = live & !fresh;
        float vI = 0.0f, vJ = 0.0f, vL = 0.0f;
        uint64_t rb = kNone, kbI = kNone, kbJ = kNone, kbL = kNone;
        if (scan) {
            vI = row[I];
            vJ = row[J];
            vL = row[Ls];
            rb = rowbest[r];
            kbI = bm[r * NB + bI];
            kbJ = bm[r * NB + bJ];
            kbL = bm[r * NB + (Ls >> sh)];
        } else if (fresh) {
            vI = agent_load(prev + I);
            vJ = agent_load(prev + J);
        }
        auto stale = [&](uint64_t k) {
            const unsigned lq = key_label(k);
            return (lq == i) | (lq == j);
        };
        const bool useJ = bJ != bI, useL = moved & (bL != bI) & (bL != bJ);  // uniform
        // (a block without slots I and J caches neither's label)
        const bool sI = scan & stale(kbI), sJ = scan & useJ & stale(kbJ);
        const uint64_t mI = __ballot(sI), mJ = __ballot(sJ);
        const int nI = __popcll(mI), n_items = nI + __popcll(mJ);
        if (n_items > 0) {
            const uint64_t below = (1ull << lane) - 1ull;
            if (sI) items[__popcll(mI & below)] = ((unsigned)r << 16) | (unsigned)bI;
            if (sJ) items[nI + __popcll(mJ & below)] = ((unsigned)r << 16) | (unsigned)bJ;
            wave_lds_sync();
            for (int base = 0; base < n_items; base += 4 * kUnroll) {
                int at[kUnroll], c0[kUnroll];
                const float* src[kUnroll];
                float4 x4[kUnroll];
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    if (base + 4 * u >= n_items) break;  // uniform
                    const int it = base + 4 * u + quarter;
                    const unsigned e = items[min(it, n_items - 1)];
                    const int rr = (int)(e >> 16), b = (int)(e & 0xFFFFu);
                    at[u] = it < n_items ? rr * NB + b : -1;
                    src[u] = D + rr * step;
                    c0[u] = (b << sh) + sub * 4;
                    x4[u] = *reinterpret_cast<const float4*>(src[u] + c0[u]);
                }
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    if (base + 4 * u >= n_items) break;
                    QuadMin m = {kFltMax, ~0u};
                    auto take = [&](const float4 v, int c) {
                        float x[4] = {v.x, v.y, v.z, v.w};
                        const int dI = I - c, dJ = J - c;  // I and J are taken out
#pragma unroll
                        for (int q = 0; q < 4; ++q) x[q] = ((dI == q) | (dJ == q)) ? kInf : x[q];
                        quad_take(m, x, label, c);
                    };
                    take(x4[u], c0[u]);
                    if constexpr (WIDE)
                        for (int c = 64; c < (1 << sh); c += 64)
                            if (c0[u] + c < (int)ld)
                                take(*reinterpret_cast<const float4*>(src[u] + c0[u] + c), c0[u] + c);
                    const uint64_t k = quad_key16(m);
                    if (sub == 15 && at[u] >= 0) bm[at[u]] = k;
                }
            }
            wave_lds_sync();
        }
        // the row's new entries and caches
        uint64_t out = kNone;
        bool again = false;  // the row's minimum has to be taken from its blocks
        if (live) {
            uint64_t kI = kNone, kL = kNone;
            float nv = 0.0f;
            if (!none) {
                nv = merge_rule(RULE, si, sj, sj, dij, vI, vJ);
                kI = row_key(nv, i);
                agent_store(next + p, nv);
            }
            if (scan) {
                if (!none) row[I] = nv;
                row[J] = kInf;  // gone: never taken again
                if (moved && p != L) kL = row_key(vL, j);
                // the entry of L, cached under its old index, comes back as kL
                auto block = [&](int b, uint64_t k) {
                    k = (moved & (key_label(k) == last)) ? kNone : k;
                    k = lesser(k, b == bI ? kI : kNone);
                    k = lesser(k, b == bL ? kL : kNone);
                    bm[r * NB + b] = k;
                };
                if (n_items > 0) {
                    kbI = bm[r * NB + bI];
                    kbJ = bm[r * NB + bJ];
                    kbL = bm[r * NB + (Ls >> sh)];
                }
                block(bI, kbI);
                if (useJ) block(bJ, kbJ);
                if (useL) block(bL, kbL);
                const uint64_t cand = lesser(kI, kL);
                const bool srb = stale(rb);
                again = (rb == kAgain) | (srb & (cand > rb));
                rb = (srb | (moved & (key_label(rb) == last))) ? kNone : rb;
                rb = lesser(rb, cand);
                if (!again) rowbest[r] = rb;
                out = rb;
            } else {
                out = kI;
            }
        } else if (own & ((p == I) | (p == J))) {
            rowbest[r] = kNone;
        }
        uint64_t mA = __ballot(again);
        if (mA) {
            wave_lds_sync();
            while (mA) {  // four rows at a time, 16 lanes each
                int src = -1;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int f = mA ? __ffsll((unsigned long long)mA) - 1 : -1;
                    if (u == quarter) src = f;
                    if (mA) mA &= mA - 1ull;
                }
                const int rr = src * W + w;
                const uint64_t k = row_min16(rr, src >= 0);
                if (sub == 15 && src >= 0) rowbest[rr] = k;
            }
            wave_lds_sync();
            if (again) out = rowbest[r];
        }
        out = min64_u64(published(out, p == L ? j : lp));
        if (lane == 0) gbest[w] = out;
        if (t == 0) agent_store(a.slots + (size_t)((s + 2) % 3) * G + g, (uint64_t)0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the merged row's entries are out before the candidate
        __syncthreads();
        if (w == 0 && s < n - 2) {
            const uint64_t k = first_min(gbest);
            if (lane == 0) agent_store(a.slots + (size_t)((s + 1) % 3) * G + g, k);
        }
        if (t == T - 1) {
            if (g == 0) {
                a.mi[s] = i;
                a.mj[s] = j;
                a.md[s] = dij;
            }
            label[J] = (uint16_t)kDead;
            if (moved) {
                label[L] = (uint16_t)j;
                slot[j] = (uint16_t)L;
            }
            sizes[i] = sj + si;
        }
        // the row merged in the step before joins the matrix; its own minimum
        // is taken in the next step.  Labels may or may not show this merge yet.
        if (pend >= 0 && pend != I && pend != J) {
            const int rr = pend / G;
            float* dst = D + rr * step;
            const float nvp = none ? 0.0f : agent_load(next + pend);
            // columns in runs of 64 per 16 lanes, kCopy of them in flight
            const int runs = (int)(ld >> 6), per = 1 << (sh - 6);  // per: runs of a block
            for (int base = (w * 4 + quarter) * per; base - quarter * per < runs; base += W * 4 * kCopy * per) {
                float2 y[kCopy][2];
#pragma unroll
                for (int u = 0; u < kCopy; ++u) {
                    if constexpr (!WIDE) {
                        const int c = min(base + u * W * 4, runs - 1) * 64 + sub * 4;
                        y[u][0] = prev_pair(c);
                        y[u][1] = prev_pair(c + 2);
                    }
                }
#pragma unroll
                for (int u = 0; u < kCopy; ++u) {
                    const int first = base + u * W * 4 * per;
                    QuadMin m = {kFltMax, ~0u};
                    for (int q = first; q < min(first + per, runs); ++q) {
                        const int c = q * 64 + sub * 4;
                        if constexpr (WIDE) {
                            y[u][0] = prev_pair(c);
                            y[u][1] = prev_pair(c + 2);
                        }
                        const ushort4 l4 = *reinterpret_cast<const ushort4*>(label + c);
                        const unsigned ls[4] = {l4.x, l4.y, l4.z, l4.w};
                        float x[4] = {y[u][0].x, y[u][0].y, y[u][1].x, y[u][1].y};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int q2 = c + e;
                            x[e] = ((q2 == I) & !none) ? nvp : x[e];
                            x[e] = ((q2 == pend) | (q2 == J) | ((ls[e] == kDead) & (q2 != L))) ? kInf : x[e];
                            const unsigned l = ((q2 == L ? j : ls[e]) << 1) | (__float_as_uint(x[e]) >> 31);
                            const bool better = (x[e] < m.v) | ((x[e] == m.v) & (l < m.l));
                            m.v = better ? x[e] : m.v;
                            m.l = better ? l : m.l;
                        }
                        *reinterpret_cast<float4*>(dst + c) = make_float4(x[0], x[1], x[2], x[3]);
                    }
                    const uint64_t k = quad_key16(m);
                    if (sub == 15 && first < runs) bm[rr * NB + first / per] = k;
                }
            }
            if (t == 0) rowbest[rr] = kAgain;
        }
        pend = (!none && I % G == g) ? I : -1;
    }
}

// Dense symmetric matrix from the packed triangle, one 64 x 64 tile (tr <= tc)
// per work-group: rows are read as the triangle holds them and the mirrored
// tile goes out through LDS, so every access is a run of 256 bytes.  Block 0
// also clears the exchange words.
__global__ __launch_bounds__(256) void agglom_init_kernel(const float* __restrict__ up, int n, int ld, int T,
                                                          float* __restrict__ D, unsigned* __restrict__ zero,
                                                          int n_zero)
{
    __shared__ float tile[64][65];
    const float kInf = __builtin_inff();
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < n_zero; k += 256) zero[k] = 0u;
    const int b = blockIdx.x;
    auto first = [T](int r) { return (int64_t)r * T - (int64_t)r * (r - 1) / 2; };
    int tr = (int)floor(((2.0 * T + 1.0) - sqrt((2.0 * T + 1.0) * (2.0 * T + 1.0) - 8.0 * b)) * 0.5);
    while (tr > 0 && first(tr) > b) --tr;
    while (tr + 1 < T && first(tr + 1) <= b) ++tr;
    const int tc = tr + (int)(b - first(tr));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = tc * 64 + lane;
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int64_t r = tr * 64 + w * 16 + k;
        v[k] = r < n && c < n && c > r ? up[r * n - r * (r + 1) / 2 + (c - r - 1)] : kInf;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) tile[w * 16 + k][lane] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int a = w * 16 + k;
        const float x = tr != tc ? tile[a][lane] : a > lane ? tile[lane][a] : a < lane ? tile[a][lane] : kInf;
        if (tr * 64 + a < n) D[(int64_t)(tr * 64 + a) * ld + c] = x;
        if (tr != tc && tc * 64 + a < n) D[(int64_t)(tc * 64 + a) * ld + tr * 64 + lane] = tile[lane][a];
    }
}

}  // namespace

// Work-groups: one per kRowsWanted rows (300 elements: 1.28 ms with 8, 1.24
// with 16, 1.31 with 32; 1000: 5.1 with 16, 4.7 with 32, 5.0 with 128) while
// there are CUs, of which one in eight is left to others: a work-group's LDS (134 KB
// at 10,000 elements) keeps most other kernels off its CU until the loop ends,
// and a launch goes to every shader engine (8 CUs) in turn, so with less than
// one CU of each free it waits.  An all-vs-all of 400 x 100 in another context,
// 45 us alone, took up to 71 ms beside 10,000 elements on 256 or 232 CUs and
// takes up to 0.2 on 224, which costs the loop 1 % (71.5 -> 72.2 ms; 12,100
// elements 98.3 -> 100.6, 15,200 165 -> 172; 15,800, whose blocks widen for it,
// 174 -> 240).  Blocks are 64 columns (one
// 16-byte load of 16 lanes), wider only where the cached minima would not fit
// the LDS: 128 from 11,201 elements, 256 from 13,601, 512 from 15,697.
bool agglom_plan(int n, int n_cu, AgglomPlan* out)
{
    if (n < 2 || n > kMaxElements) return false;
    AgglomPlan p;
    p.groups = std::max(1, std::min(std::min(n_cu - n_cu / 8, 64 * kWaves), n / kRowsWanted));
    p.rows = (n + p.groups - 1) / p.groups;
    if (p.rows > 64 * kWaves) return false;
    for (p.block_shift = 6; p.block_shift <= 9; ++p.block_shift) {
        p.n_blocks = (n + (1 << p.block_shift) - 1) >> p.block_shift;
        const size_t n4 = (size_t)(n + 3) / 4 * 4, cap = (size_t)p.n_blocks << p.block_shift;
        p.lds = (size_t)p.rows * p.n_blocks * 8 + (size_t)p.rows * 8 + 2 * kWaves * 8 + cap * 2 + n4 * 2 + n4 * 4 +
                (size_t)kWaves * kWaveItems * 4 + 16;
        if (p.lds <= kLdsBytes) {
            *out = p;
            return true;
        }
    }
    return false;
}

void launch_agglom_init(const float* up, int n, int ld, float* D, unsigned* zero, int n_zero, hipStream_t s)
{
    const int T = (n + 63) / 64;
    agglom_init_kernel<<<T * (T + 1) / 2, 256, 0, s>>>(up, n, ld, T, D, zero, n_zero);
}

namespace {
template <bool WIDE>
const void* agglom_entry(int rule)
{
    switch (rule) {
    case 0: return reinterpret_cast<const void*>(&agglom_kernel<WIDE, 0>);
    case 1: return reinterpret_cast<const void*>(&agglom_kernel<WIDE, 1>);
    case 2: return reinterpret_cast<const void*>(&agglom_kernel<WIDE, 2>);
    case 3: return reinterpret_cast<const void*>(&agglom_kernel<WIDE, 3>);
    case 4: return reinterpret_cast<const void*>(&agglom_kernel<WIDE, 4>);
    default: return reinterpret_cast<const void*>(&agglom_kernel<WIDE, 5>);
    }
}
}  // namespace

// As exact_init; where the limit is not taken the launch is refused.
void agglom_init()
{
    for (int rule = 0; rule < 6; ++rule)
        for (const void* f : {agglom_entry<false>(rule), agglom_entry<true>(rule)})
            if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess)
                (void)hipGetLastError();
}

hipError_t launch_agglom(const AgglomPlan& p, AgglomArgs a, hipStream_t s)
{
    a.rows = p.rows;
    a.n_blocks = p.n_blocks;
    a.block_shift = p.block_shift;
    const void* f = p.block_shift == 6 ? agglom_entry<false>(a.rule) : agglom_entry<true>(a.rule);
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(f, dim3(p.groups), dim3(64 * kWaves), args, (unsigned)p.lds, s);
}

}  // namespace bs
