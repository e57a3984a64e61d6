// gram_split.hpp -- one 32 x 32 tile of the Gram kernels by a work-group of
// four waves, for the last, partly filled round of a launch's 64 x 64 tiles.
#pragma once

#include "gram_tile.hpp"

namespace bs {

// Operand words of one atom block for the wave of row coordinate c: words
// 2c, 2c + 1 of the row block, all six of the column block.
struct SplitRegs {
    uint4 a[2], b[6];
};

template <int MODE>
__device__ __forceinline__ void split_load(const uint4* __restrict__ A, const uint4* __restrict__ B, int c, int lane,
                                           SplitRegs& r)
{
#pragma unroll
    for (int u = 0; u < 2; ++u)
        r.a[u] = A[MODE == kGramBF16x3 ? (2 * c + u) * 64 + lane : c * 128 + 2 * lane + u];
#pragma unroll
    for (int u = 0; u < 6; ++u)
        r.b[u] = B[MODE == kGramBF16x3 ? u * 64 + lane : (u >> 1) * 128 + 2 * lane + (u & 1)];
}

// The products of row coordinate c with the three column coordinates, each
// accumulator in mfma_regs' order: the same sums bit for bit.
template <int MODE>
__device__ __forceinline__ void split_mfma(const SplitRegs& r, f32x16 (&acc)[3])
{
    if constexpr (MODE == kGramBF16x3) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(r.a[0]), as_bf16x8(r.b[2 * d]), acc[d], 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(r.a[0]), as_bf16x8(r.b[2 * d + 1]), acc[d], 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(r.a[1]), as_bf16x8(r.b[2 * d]), acc[d], 0, 0, 0);
    } else {
        const float fa[8] = {__uint_as_float(r.a[0].x), __uint_as_float(r.a[0].y), __uint_as_float(r.a[0].z),
                             __uint_as_float(r.a[0].w), __uint_as_float(r.a[1].x), __uint_as_float(r.a[1].y),
                             __uint_as_float(r.a[1].z), __uint_as_float(r.a[1].w)};
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const uint4 w = r.b[2 * d + (s >> 2)];
                const unsigned u = (s & 3) == 0 ? w.x : (s & 3) == 1 ? w.y : (s & 3) == 2 ? w.z : w.w;
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[s], __uint_as_float(u), acc[d], 0, 0, 0);
            }
    }
}

// LDS: three stages of one atom block's row and column operands (12 KiB each),
// which the nine accumulators of the tile's pairs take over.
union SplitLds {
    uint4 ring[3][2][kPanelBlockU4];
    float e[9][1024];
};

// Roles 0..2 run the products of one row coordinate each, role 3 streams the
// operands: the products' waves issue no memory access and hold three
// accumulators instead of nine.  `turn` rotates the roles over the waves, so
// that two such tiles on a CU do not leave the same SIMD without products.
// The accumulators then go through LDS, and all 256 threads solve four pairs
// each, two at a time: pair k of thread t is row t / 32 + 8 k, column t % 32.
// What bounds a 64 x 64 tile alone on its CU is latency: 16 FP64 solves per
// lane with one wave per SIMD (8 of its 14.5 us at 150 atoms), then the K
// loop of nine accumulators per SIMD.  Here both are shared by four CUs: an
// ensemble of 500 x 150 took 17.6 us in one launch of 64 x 64 tiles and takes
// 9.2 (bf16x3; FP32 34.4 and 14.1).  Each pair's sums, solve and flag are the
// 64 x 64 tile's, bit for bit.
// STATS: the tile's 128 keys (row and column minima and maxima) go to
// a.stats_part; the key array is in LDS behind the accumulators.
template <int MODE, bool STATS>
__device__ __forceinline__ void gram_split32(const GramArgs& a, int tr, int tc, char* smem, int turn, int t)
{
    SplitLds& lds = *reinterpret_cast<SplitLds*>(smem);
    unsigned(*skeys)[33] = reinterpret_cast<unsigned(*)[33]>(smem + sizeof(SplitLds));
    const int lane = t & 63;
    // the tile's row and column keys within its 64 x 64 tile's two banks
    unsigned* rkeys = nullptr;
    unsigned* ckeys = nullptr;
    if constexpr (STATS) {
        const int r6 = tr >> 1, c6 = tc >> 1;
        unsigned* p = a.stats_part + ((int64_t)r6 * a.stats_T - (int64_t)r6 * (r6 - 1) / 2 + (c6 - r6)) * 512;
        rkeys = p + 256 * (tc & 1) + 32 * (tr & 1);
        ckeys = p + 256 * (tr & 1) + 128 + 32 * (tc & 1);
    }
    if (tr * 32 >= a.n_rows || tc * 32 >= a.n_cols || (a.triangle && tr > tc)) {
        if constexpr (STATS)
            if (t < 32) {
                rkeys[t] = ckeys[t] = 0xFFFFFFFFu;
                rkeys[64 + t] = ckeys[64 + t] = 0u;
            }
        return;
    }
    const int role = __builtin_amdgcn_readfirstlane((t >> 6) + turn) & 3;
    const int n_kblk = a.n_kblk, last = n_kblk - 1;
    if (role == 3) {
        const uint4* sa = static_cast<const uint4*>(a.panels_a) + (int64_t)tr * n_kblk * kPanelBlockU4 + lane;
        const uint4* sb = static_cast<const uint4*>(a.panels_b) + (int64_t)tc * n_kblk * kPanelBlockU4 + lane;
        auto issue = [&](int kb, int st) {
            const int64_t o = (int64_t)min(kb, last) * kPanelBlockU4;
#pragma unroll
            for (int u = 0; u < 6; ++u) {
                BS_GLOAD_LDS(sa + o + u * 64, &lds.ring[st][0][u * 64]);
                BS_GLOAD_LDS(sb + o + u * 64, &lds.ring[st][1][u * 64]);
            }
        };
        issue(0, 0);
        issue(1, 1);
        issue(2, 2);
        BS_WAIT_VMCNT(24);
        __builtin_amdgcn_s_barrier();  // block 0 is in LDS
        int st = 0;
        for (int k = 0; k < n_kblk; ++k) {
            BS_WAIT_VMCNT(12);
            __builtin_amdgcn_s_barrier();  // block k + 1 is in LDS, block k in the others' registers
            issue(k + 3, st);
            st = st == 2 ? 0 : st + 1;
        }
        BS_WAIT_VMCNT(0);  // no load may still write the LDS the accumulators take
        __builtin_amdgcn_s_barrier();
    } else {
        f32x16 acc[3];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[d][r] = 0.0f;
        SplitRegs ra, rb;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        split_load<MODE>(lds.ring[0][0], lds.ring[0][1], role, lane, ra);
        int st = 0;
        auto step = [&](const SplitRegs& cur, SplitRegs& nxt) {
            st = st == 2 ? 0 : st + 1;
            BS_WAIT_LDS0();
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            split_load<MODE>(lds.ring[st][0], lds.ring[st][1], role, lane, nxt);
            split_mfma<MODE>(cur, acc);
        };
        for (int k = 0; k < n_kblk; k += 2) {
            step(ra, rb);
            if (k + 1 >= n_kblk) break;
            step(rb, ra);
        }
        BS_WAIT_LDS0();
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                lds.e[3 * role + d][(8 * (r / 4) + 4 * (lane >> 5) + r % 4) * 32 + (lane & 31)] = acc[d][r];
    }
    // constants straight from memory: the loads cover the exchange's barrier
    const int jl = t & 31, j = tc * 32 + jl;
    const bool jok = j < a.n_cols;
    const EpilogueLimits& lim = a.lim;
    double cj[kNumConsts];
#pragma unroll
    for (int q = 0; q < kNumConsts; ++q) cj[q] = a.consts_b[(int64_t)q * a.ldb + min(j, a.n_cols - 1)];
    __syncthreads();

    uint32_t flagged = 0;
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
        double c[2][kNumConsts], E[2][9];
        PairSolve o[2];
        bool flag[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int il = (t >> 5) + 8 * (k + p);
#pragma unroll
            for (int q = 0; q < kNumConsts; ++q)
                c[p][q] = a.consts_a[(int64_t)q * a.lda + min(tr * 32 + il, a.n_rows - 1)];
#pragma unroll
            for (int q = 0; q < 9; ++q) E[p][q] = (double)lds.e[q][il * 32 + jl];
        }
        solve_pairs<2>(E, c, cj, lim, o, flag);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int il = (t >> 5) + 8 * (k + p), i = tr * 32 + il;
            const bool ok = jok && i < a.n_rows && (!a.triangle || i < j);
            const int64_t oi = a.triangle ? tri_index(a.n_rows, i, j) : (int64_t)i * a.out_ld + j;
            if (!STATS && a.out_f64) {
                if (ok) static_cast<double*>(a.out)[oi] = sqrt(o[p].rmsd2_L * lim.inv_L);
            } else {
                const float v = __builtin_amdgcn_sqrtf((float)(o[p].rmsd2_L * lim.inv_L));
                if (ok) static_cast<float*>(a.out)[oi] = v;
                if constexpr (STATS)
                    skeys[il][jl] = ok && !flag[p] && v == v ? fkey(__float_as_uint(v)) : 0xFFFFFFFFu;
            }
            flagged |= (uint32_t)(ok & flag[p]) << (k + p);
        }
    }
    flag_pairs<4>(a, flagged, lane, [&](int k) {
        const int i = tr * 32 + (t >> 5) + 8 * k;
        return a.triangle ? tri_index(a.n_rows, i, j) : (int64_t)i * a.out_ld + j;
    });
    if constexpr (STATS) {
        __syncthreads();
        // tile row r and tile column r: eight threads of four entries each
        const int r = t >> 3, q = t & 7;
        unsigned lo = 0xFFFFFFFFu, hi = 0u, clo = 0xFFFFFFFFu, chi = 0u;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const unsigned kr = skeys[r][q * 4 + c], kc = skeys[q * 4 + c][r];
            lo = min(lo, kr);
            hi = max(hi, kr == 0xFFFFFFFFu ? 0u : kr);
            clo = min(clo, kc);
            chi = max(chi, kc == 0xFFFFFFFFu ? 0u : kc);
        }
#pragma unroll
        for (int m = 1; m <= 4; m <<= 1) {
            lo = min(lo, (unsigned)__shfl_xor((int)lo, m));
            hi = max(hi, (unsigned)__shfl_xor((int)hi, m));
            clo = min(clo, (unsigned)__shfl_xor((int)clo, m));
            chi = max(chi, (unsigned)__shfl_xor((int)chi, m));
        }
        if (q == 0) {
            rkeys[r] = lo;
            rkeys[64 + r] = hi;
            ckeys[r] = clo;
            ckeys[64 + r] = chi;
        }
    }
}

}  // namespace bs
