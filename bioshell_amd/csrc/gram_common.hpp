// gram_common.hpp -- pieces shared by the Gram kernels.
#pragma once

#include "exact_solve.hpp"
#include "kernels.hpp"
#include "qcp.hpp"
#include "wave.hpp"

namespace bs {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kXcd = 8;  // MI355X: work-group ids are dealt to 8 XCDs round-robin

__device__ inline int64_t tri_index(int64_t n, int64_t i, int64_t j)
{
    return i * n - i * (i + 1) / 2 + (j - i - 1);
}

__device__ inline bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// One atom block of the nine 32x32 accumulators of a wave: rows from the A
// stage block (32 conformations), columns from the B stage block.
template <int MODE>
__device__ __forceinline__ void mfma_block(const uint4* __restrict__ A, const uint4* __restrict__ B,
                                           int lane, f32x16 (&acc)[9])
{
    if constexpr (MODE == kGramBF16x3) {
        bf16x8 ah[3], al[3], bh[3], bl[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            ah[c] = as_bf16x8(A[(2 * c) * 64 + lane]);
            al[c] = as_bf16x8(A[(2 * c + 1) * 64 + lane]);
            bh[c] = as_bf16x8(B[(2 * c) * 64 + lane]);
            bl[c] = as_bf16x8(B[(2 * c + 1) * 64 + lane]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int d = 0; d < 3; ++d)
                acc[3 * c + d] =
                    __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], bh[d], acc[3 * c + d], 0, 0, 0);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int d = 0; d < 3; ++d)
                acc[3 * c + d] =
                    __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], bl[d], acc[3 * c + d], 0, 0, 0);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int d = 0; d < 3; ++d)
                acc[3 * c + d] =
                    __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[c], bh[d], acc[3 * c + d], 0, 0, 0);
    } else {
        float fa[3][8], fb[3][8];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const uint4 a0 = A[c * 128 + 2 * lane], a1 = A[c * 128 + 2 * lane + 1];
            const uint4 b0 = B[c * 128 + 2 * lane], b1 = B[c * 128 + 2 * lane + 1];
            fa[c][0] = __uint_as_float(a0.x); fa[c][1] = __uint_as_float(a0.y);
            fa[c][2] = __uint_as_float(a0.z); fa[c][3] = __uint_as_float(a0.w);
            fa[c][4] = __uint_as_float(a1.x); fa[c][5] = __uint_as_float(a1.y);
            fa[c][6] = __uint_as_float(a1.z); fa[c][7] = __uint_as_float(a1.w);
            fb[c][0] = __uint_as_float(b0.x); fb[c][1] = __uint_as_float(b0.y);
            fb[c][2] = __uint_as_float(b0.z); fb[c][3] = __uint_as_float(b0.w);
            fb[c][4] = __uint_as_float(b1.x); fb[c][5] = __uint_as_float(b1.y);
            fb[c][6] = __uint_as_float(b1.z); fb[c][7] = __uint_as_float(b1.w);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    acc[3 * c + d] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[c][s], fb[d][s],
                                                                          acc[3 * c + d], 0, 0, 0);
    }
}

// Row of packed-triangle position o (row-major upper triangle of n, i < j).
__device__ inline int tri_row(int64_t o, int n)
{
    const double b = 2.0 * n - 1.0;
    int i = (int)floor((b - sqrt(b * b - 8.0 * (double)o)) * 0.5);
    auto start = [n](int64_t r) { return r * n - r * (r + 1) / 2; };
    while (i > 0 && start(i) > o) --i;
    while (start(i + 1) <= o) ++i;
    return i;
}

// One pair for FP64 re-evaluation: coordinates, centroids, atom count.
struct PairRef {
    const double* x;
    const double* y;
    const double* cx;
    const double* cy;
    int L;  // 0: no pair
};

// Chains of up to this many atoms are summed by 8 lanes per pair, longer ones
// by a wave per pair (the sums' order, so the result, depends on L alone).
constexpr int kShortChain = 64;

// The sums one pair's QCP needs: the covariance and both inner products.
struct PairSums {
    double m[9], ga, gb;
};

__device__ __forceinline__ void add_atom(PairSums& s, double a0, double a1, double a2, double b0, double b1, double b2)
{
    s.m[0] += a0 * b0; s.m[1] += a0 * b1; s.m[2] += a0 * b2;
    s.m[3] += a1 * b0; s.m[4] += a1 * b1; s.m[5] += a1 * b2;
    s.m[6] += a2 * b0; s.m[7] += a2 * b1; s.m[8] += a2 * b2;
    s.ga += a0 * a0 + a1 * a1 + a2 * a2;
    s.gb += b0 * b0 + b1 * b1 + b2 * b2;
}

// Atoms k0, k0 + STRIDE, k0 + 2 STRIDE and k0 + 3 STRIDE of a pair (those below
// L), centred: all 24 loads in flight at once, a missing atom adding zeros.
template <int STRIDE>
__device__ __forceinline__ void add_atoms(PairSums& s, const double* __restrict__ x, const double* __restrict__ y,
                                          const double (&c)[6], int k0, int L)
{
    double a[4][6];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int k = min(k0 + STRIDE * u, L - 1);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            a[u][d] = x[3 * k + d];
            a[u][3 + d] = y[3 * k + d];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        double v[6];
#pragma unroll
        for (int d = 0; d < 6; ++d) v[d] = k0 + STRIDE * u < L ? a[u][d] - c[d] : 0.0;
        add_atom(s, v[0], v[1], v[2], v[3], v[4], v[5]);
    }
}

// Sum over each group of 8 lanes (all active), in every lane.
__device__ __forceinline__ double oct_sum(double v)
{
    v += dpp_f64<0xB1, 0xF, true>(v);   // quad_perm [1, 0, 3, 2]
    v += dpp_f64<0x4E, 0xF, true>(v);   // quad_perm [2, 3, 0, 1]
    v += dpp_f64<0x141, 0xF, true>(v);  // row_half_mirror
    return v;
}

__device__ __forceinline__ const double* shfl_ptr(const double* p, int src)
{
    const uint64_t b = (uint64_t)p;
    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)b, src), hi = (uint32_t)__shfl((int)(uint32_t)(b >> 32), src);
    return reinterpret_cast<const double*>(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ const double* lane_ptr(const double* p, int src)
{
    const uint64_t b = (uint64_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
    return reinterpret_cast<const double*>(((uint64_t)hi << 32) | lo);
}

// FP64 cRMSD of up to 64 pairs from raw coordinates, one per lane (all lanes
// active; the result of a lane without a pair means nothing): centring on the
// fly, then the textbook QCP with the near-degenerate polish.
//
// What a pair costs a wave is the cross-lane sums and the solve (some 5,000
// cycles of dependent FP64, mostly divisions), not its products.  The pairs
// are therefore summed by 8 lanes each (3 exchange steps instead of 6, eight
// pairs at a time) or one after the other by the wave, each lane keeps its own
// pair's sums, and the solve runs once for all 64.  One pair at a time took
// 6.5 ns per pair chip-wide whatever its length.
__device__ inline double fallback_pairs(const PairRef& p, int lane)
{
    PairSums mine{};
    const int sub = lane & 7;
    const uint64_t shorts = __ballot(p.L > 0 && p.L <= kShortChain);
    if (shorts) {
#pragma unroll 1
        for (int s = 0; s < 8; ++s) {
            if (!((shorts >> s) & 0x0101010101010101ull)) continue;  // pair s of each group of 8 lanes
            const int src = (lane & ~7) + s;
            const int Ls = __shfl(p.L, src);
            const int L = Ls <= kShortChain ? Ls : 0;
            const double* x = shfl_ptr(p.x, src);
            const double* y = shfl_ptr(p.y, src);
            const double* cx = shfl_ptr(p.cx, src);
            const double* cy = shfl_ptr(p.cy, src);
            PairSums t{};
            if (L > 0) {
                const double c[6] = {cx[0], cx[1], cx[2], cy[0], cy[1], cy[2]};
#pragma unroll 1
                for (int k0 = sub; k0 < L; k0 += 32) add_atoms<8>(t, x, y, c, k0, L);
            }
            const bool keep = sub == s;
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                const double v = oct_sum(t.m[q]);
                mine.m[q] = keep ? v : mine.m[q];
            }
            const double va = oct_sum(t.ga), vb = oct_sum(t.gb);
            mine.ga = keep ? va : mine.ga;
            mine.gb = keep ? vb : mine.gb;
        }
    }
    uint64_t longs = __ballot(p.L > kShortChain);
#pragma unroll 1
    while (longs) {
        const int src = __ffsll((unsigned long long)longs) - 1;
        longs &= longs - 1;
        const int L = __builtin_amdgcn_readlane(p.L, src);
        const double* x = lane_ptr(p.x, src);
        const double* y = lane_ptr(p.y, src);
        const double* cx = lane_ptr(p.cx, src);
        const double* cy = lane_ptr(p.cy, src);
        const double c[6] = {cx[0], cx[1], cx[2], cy[0], cy[1], cy[2]};
        PairSums t{};
#pragma unroll 1
        for (int k0 = lane; k0 < L; k0 += 256) add_atoms<64>(t, x, y, c, k0, L);
        const bool keep = lane == src;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const double v = wave_sum(t.m[q]);
            mine.m[q] = keep ? v : mine.m[q];
        }
        const double va = wave_sum(t.ga), vb = wave_sum(t.gb);
        mine.ga = keep ? va : mine.ga;
        mine.gb = keep ? vb : mine.gb;
    }
    return exact_rmsd(mine.m, mine.ga, mine.gb, max(p.L, 1), p.L > 0);
}

// Walks a wave through the flagged outputs, up to 64 at a time: its share of
// the queued entries list[0 .. m), then, where the bitmap is scanned too, the
// set bits of 64 words at a time, whose positions go through LDS (2048 entries
// of this wave at `slots`).  next() gives each lane an output or -1 (no pair
// in the lane), the first eight of a trip to different groups of 8 lanes, and
// returns false (in every lane) when nothing is left.
struct FlagCursor {
    const int64_t* list;
    uint32_t* bits;  // or null
    uint16_t* slots;
    int64_t n_words, w0;
    int m, k0, step, n_waves, lane, per, slot, total, at;

    // list_wave of list_waves share the list, wave of n_waves_ the bitmap
    __device__ FlagCursor(const int64_t* list_, uint32_t m_, int list_wave, int list_waves, uint32_t* bits_,
                          int64_t n_words_, int wave, int n_waves_, uint16_t* slots_, int lane_)
        : list(list_), bits(bits_), slots(slots_), n_words(n_words_), w0((int64_t)wave * 64), m((int)m_),
          n_waves(n_waves_), lane(lane_), slot((lane_ & 7) * 8 + (lane_ >> 3)), total(0), at(0)
    {
        per = (int)min(64u, (m_ + list_waves - 1) / (uint32_t)list_waves);
        k0 = list_wave * per;
        step = list_waves * per;
    }

    __device__ bool next(int64_t& o)
    {
        o = -1;
        if (k0 < m) {
            if (slot < per && k0 + slot < m) o = list[k0 + slot];
            k0 += step;
            return true;
        }
        while (at >= total) {
            if (!bits || w0 >= n_words) return false;
            uint32_t word = w0 + lane < n_words ? bits[w0 + lane] : 0u;
            if (word) bits[w0 + lane] = 0u;
            const int cnt = __popc(word);
            int incl = cnt;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            total = __builtin_amdgcn_readlane(incl, 63);
            int pos = incl - cnt;
            wave_lds_sync();  // the previous entries are read
            while (word) {
                slots[pos++] = (uint16_t)(lane * 32 + __ffs(word) - 1);
                word &= word - 1u;
            }
            wave_lds_sync();
            at = 0;
            w0 += (int64_t)n_waves * 64;
        }
        if (at + slot < total) o = (w0 - (int64_t)n_waves * 64) * 32 + slots[at + slot];
        at += 64;
        return true;
    }
};

// Marks a wave's flagged pairs for FP64 re-evaluation (all lanes active; bit r
// of `flagged`: the lane's pair r, output out_index(r), which grows by one
// from lane to lane within a half-wave): queued in the list while it has room,
// else as bits in the bitmap.  One atomic per wave reserves the places and two
// per half-wave set a row's bits: one atomic per pair took 0.32 of the 0.40 ms
// of a launch of 2000 x 20 atoms that flags 58 % of its pairs.
template <int NR, class F>
__device__ __forceinline__ void flag_pairs(const GramArgs& a, uint32_t flagged, int lane, F out_index)
{
    if (!__any(flagged != 0u)) return;
    uint32_t base = 0, cap = 0;
    if (a.flag_list) {
        uint32_t total = 0;
#pragma unroll 1
        for (int r = 0; r < NR; ++r) total += (uint32_t)__popcll(__ballot((flagged >> r) & 1u));
        const int k = blockIdx.x % kFlagLists;
        int64_t* list = a.flag_list + (int64_t)k * a.flag_cap;
        if (lane == 0) base = atomicAdd(a.flag_ctl + 16 * k, total);
        base = __builtin_amdgcn_readfirstlane(base);
        cap = (uint32_t)a.flag_cap;
        if (base < cap) {
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                const bool f = (flagged >> r) & 1u;
                const uint64_t m = __ballot(f);
                const uint32_t pos = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                base += (uint32_t)__popcll(m);
                if (f && pos < cap) {
                    list[pos] = out_index(r);
                    flagged &= ~(1u << r);
                }
            }
            if (base <= cap) return;
        }
    }
#pragma unroll 1
    for (int r = 0; r < NR; ++r) {
        const uint64_t m = __ballot((flagged >> r) & 1u);
        if (!m) continue;
        const uint32_t row = (uint32_t)(m >> (lane & 32));
        const int64_t o = out_index(r) - (lane & 31);  // of bit 0; below 0 only where its bits are 0
        const int sh = (int)(o & 31), w = lane & 31;
        const uint32_t bits = w == 0 ? row << sh : (w == 1 && sh ? row >> (32 - sh) : 0u);
        if (bits) atomicOr(a.flag_bits + (o >> 5) + w, bits);
    }
}

}  // namespace bs
