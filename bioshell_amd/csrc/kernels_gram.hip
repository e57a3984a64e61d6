// kernels_gram.hip -- covariance as a Gram contraction on MFMA, fused with the
// FP64 shifted-QCP epilogue, plus the FP64 re-evaluation of flagged pairs.
//
// For a block of pairs (i, j) the nine residual cross-covariances
//     E_cd(i, j) = sum_k e_i,k,c * e_j,k,d          (c, d in {x, y, z})
// are nine GEMM tiles that share three row panels (e_x, e_y, e_z of the rows)
// and three column panels.  A wave owns a 32 x 32 block of pairs and keeps the
// nine 32x32 FP32 accumulators of v_mfma_f32_32x32x16_bf16 (or _32x32x2f32);
// lane l then holds column j = l % 32 and rows 8(r/4) + 4(l/32) + r%4 of all
// nine tiles, so the 3x3 matrix of every pair it owns is lane-local and the
// QCP epilogue runs without any exchange.
//
// BF16x3: operands are split e = hi + lo (two bf16) and each tile accumulates
// hi*hi + hi*lo + lo*hi in FP32.  A work-group (4 waves) covers 64 x 64 pairs;
// operand blocks (32 conformations x 16 atoms, 6 KiB) are double-buffered
// through LDS.  Work-group ids are dealt to the 8 XCDs round-robin, so the
// logical tile is taken from a contiguous per-XCD slice of a super-blocked
// order: each XCD's L2 keeps re-using the same row and column panels.
#include "gram_split.hpp"

#include <algorithm>

namespace bs {
namespace {

// One work-group per 64 x 64 tile, then one per 32 x 32 tile of the tiles past
// a.n_full (gram_full_tiles).  Work-group ids are dealt to the 8 XCDs
// round-robin, so the logical tile comes from a contiguous per-XCD slice of
// the super-blocked order.  Two work-groups share each CU, and on a SIMD one's
// MFMA phase overlaps the other's FP64 epilogue (VALU).
template <int MODE, bool STATS>
__global__ __launch_bounds__(256, 2) void gram_kernel(GramArgs a)
{
    __shared__ uint4 lds[3][4][kPanelBlockU4];  // 3 stages x (A0, A1, B0, B1) x 6 KiB
    const int wg = blockIdx.x;
    const int per = (a.n_full + kXcd - 1) / kXcd;
    if (wg < per * kXcd) {
        const int t = (wg % kXcd) * per + (wg / kXcd);
        if (t >= a.n_full) return;
        const uint32_t code = a.tiles[t];
        stamp_start(a.t_start);  // after the read, which a store before it would make per lane
        gram_tile64<MODE, true, 2, STATS>(a, (int)(code >> 16), (int)(code & 0xFFFFu), lds, (int)threadIdx.x);
        return;
    }
    const int w = wg - per * kXcd, n_quad = a.quads * (a.n_tiles - a.n_full);
    const int per_q = (n_quad + kXcd - 1) / kXcd;
    const int q = (w % kXcd) * per_q + (w / kXcd);
    if (q >= n_quad) return;
    const uint32_t code = a.tiles[a.n_full + q / a.quads];
    const int part = q % a.quads;
    stamp_start(a.t_start);
    const int tr = 2 * (int)(code >> 16) + (part >> 1), tc = 2 * (int)(code & 0xFFFFu) + (part & 1);
    gram_split32<MODE, STATS>(a, tr, tc, reinterpret_cast<char*>(lds), (w / kXcd) >> 5, (int)threadIdx.x);
}

__global__ void zero_u32_kernel(uint32_t* p, int n)
{
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v < n) p[v] = 0u;
}

__global__ void zero_words_kernel(uint4* p, int64_t n4)
{
    for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < n4; v += (int64_t)gridDim.x * 256)
        p[v] = make_uint4(0u, 0u, 0u, 0u);
}

// Queues the set bits of the flag bitmap: one thread per word; a wave scan of
// the words' bit counts and one atomic per wave give each word its slots.
// Queued bits are cleared; bits that do not fit in the list (cap entries)
// stay set for a bitmap scan.  *count receives the number of set bits.  (The
// batched pipeline's flag path; a single Gram launch queues directly.)
__global__ __launch_bounds__(256) void flag_compact_kernel(uint32_t* __restrict__ bits,
                                                           int64_t n_words,
                                                           int64_t* __restrict__ list, int cap,
                                                           uint32_t* __restrict__ count)
{
    const int lane = threadIdx.x & 63;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t base_w = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~63); base_w < n_words;
         base_w += stride) {
        const int64_t w = base_w + lane;
        uint32_t word = w < n_words ? bits[w] : 0u;
        const int p = __popc(word);
        int incl = p;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o);
            if (lane >= o) incl += t;
        }
        const int total = __shfl(incl, 63);
        if (total == 0) continue;
        uint32_t start = 0;
        if (lane == 63) start = atomicAdd(count, (uint32_t)total);
        start = __shfl(start, 63);
        int64_t pos = (int64_t)start + (incl - p);
        if (p) {
            uint32_t left = word;
            while (word) {
                const int b = __ffs(word) - 1;
                word &= word - 1u;
                if (pos < cap) {
                    list[pos] = w * 32 + b;
                    left &= ~(1u << b);
                }
                ++pos;
            }
            bits[w] = left;
        }
    }
}

// Decodes output o of a triangle (n x n, i < j) or of a dense n_rows x out_ld block.
__device__ inline void decode_output(int64_t o, int triangle, int n, int64_t out_ld, int& i, int& j)
{
    if (triangle) {
        i = tri_row(o, n);
        j = (int)(o - ((int64_t)i * n - (int64_t)i * (i + 1) / 2)) + i + 1;
    } else {
        i = (int)(o / out_ld);
        j = (int)(o - (int64_t)i * out_ld);
    }
}

// The flagged outputs of one Gram launch, up to 64 per wave at a time: the
// queued entries, work-group b taking its part of list b % kFlagLists, then,
// only when a list overflowed, a scan of the bitmap in which each wave takes 64
// words and clears them.  The last work-group to finish publishes the count
// and zeroes the other control words for the next launch; the groups count
// themselves done per list, then the lists (on one word their atomics, 9 ns
// apart, made an empty list take 3.7 us; this way 2.2).
constexpr int kResolveWaves = 4;  // per work-group

__global__ __launch_bounds__(64 * kResolveWaves) void flag_resolve_kernel(
    const double* __restrict__ xa, const double* __restrict__ ca, const double* __restrict__ xb,
    const double* __restrict__ cb, int L, uint32_t* __restrict__ ctl, const int64_t* __restrict__ list, int cap,
    uint32_t* __restrict__ bits, int64_t n_out, int triangle, int n, int64_t out_ld, void* __restrict__ out,
    int out_f64, uint32_t* h_report, unsigned* st_min, unsigned* st_max, uint64_t* clk, int ends_call)
{
    __shared__ uint16_t slots[kResolveWaves][2048];
    stamp_start(clk ? clk + kClkResolve : nullptr);
    const int lane = threadIdx.x & 63;
    const int seg = (int)blockIdx.x % kFlagLists, w = threadIdx.x >> 6;
    // read before this group counts itself done
    const uint32_t mine = lane < kFlagLists ? ctl[16 * lane] : 0u;
    const bool overflow = __any(mine > (uint32_t)cap);
    const uint32_t cnt = __builtin_amdgcn_readlane(mine, seg);
    FlagCursor cur(list + (int64_t)seg * cap, min(cnt, (uint32_t)cap), (int)blockIdx.x / kFlagLists * kResolveWaves + w,
                   (int)gridDim.x / kFlagLists * kResolveWaves, overflow ? bits : nullptr, (n_out + 31) >> 5,
                   (int)blockIdx.x * kResolveWaves + w, (int)gridDim.x * kResolveWaves, slots[w], lane);
    for (int64_t o; __builtin_expect(cur.next(o), 0);) {
        PairRef p{xa, xb, ca, cb, 0};
        int i = 0, j = 0;
        if (o >= 0 && o < n_out) {
            decode_output(o, triangle, n, out_ld, i, j);
            p = {xa + (int64_t)i * L * 3, xb + (int64_t)j * L * 3, ca + 3 * (int64_t)i, cb + 3 * (int64_t)j, L};
        }
        const double r = fallback_pairs(p, lane);
        if (!p.L) continue;
        if (out_f64) {
            static_cast<double*>(out)[o] = r;
            continue;
        }
        const float v = (float)r;
        static_cast<float*>(out)[o] = v;
        // the stored value joins both elements' keys, which only fall (rise):
        // one already beyond it needs no atomic
        if (st_min && v == v) {
            const unsigned k = fkey(__float_as_uint(v));
            if (k < st_min[i]) atomicMin(st_min + i, k);
            if (k < st_min[j]) atomicMin(st_min + j, k);
            if (k > st_max[i]) atomicMax(st_max + i, k);
            if (k > st_max[j]) atomicMax(st_max + j, k);
        }
    }
    // Every thread of the group has used its copy of the counts (no fence:
    // the reset only needs the reads done, and the next launch sees it).
    __syncthreads();
    if (threadIdx.x >= 64) return;
    uint32_t all = mine;
#pragma unroll
    for (int d = 1; d < kFlagLists; d <<= 1) all += (uint32_t)__shfl_xor((int)all, d);
    if (threadIdx.x == 0 && atomicAdd(&ctl[16 * seg + 1], 1u) == gridDim.x / kFlagLists - 1 &&
        atomicAdd(&ctl[2], 1u) == kFlagLists - 1) {
        ctl[2] = 0u;
        ctl[3] = all;
        for (int k = 0; k < kFlagLists; ++k) ctl[16 * k] = ctl[16 * k + 1] = 0u;
        if (h_report) __hip_atomic_store(h_report, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (clk) {
            const uint64_t now = wall_clock64();
            clk[kClkResolveEnd] = now;
            clk[kClkCount] = all;
            if (ends_call) clk[kClkEnd] = now;
        }
    }
}

}  // namespace

int build_tile_order(int tiles_r, int tiles_c, bool triangle, int super, uint32_t* out)
{
    int n = 0;
    const int sr_n = (tiles_r + super - 1) / super, sc_n = (tiles_c + super - 1) / super;
    for (int sr = 0; sr < sr_n; ++sr)
        for (int sc = triangle ? sr : 0; sc < sc_n; ++sc)
            for (int r = sr * super; r < min((sr + 1) * super, tiles_r); ++r)
                for (int c = sc * super; c < min((sc + 1) * super, tiles_c); ++c)
                    if (!triangle || r <= c) out[n++] = ((uint32_t)r << 16) | (uint32_t)c;
    return n;
}

// A 64 x 64 tile takes a CU about as long alone (bf16x3, 150 atoms: 14.5 us
// past the launch) as two take it together (21), so a launch's last, partly
// filled round of n_cu tiles costs as much as a full one.  As 32 x 32 tiles
// over the idle CUs it takes 6 us with one each and 12 with two, but four
// cost more than the tile they replace.  Measured on 256 CUs against 64 x 64
// tiles only (bf16x3, 100 and 260 atoms): less than one round, remainders up
// to 0.21 n_cu 1.8-2.1x faster, 0.26-0.47 1.4-1.5x, 0.53 +-3 %, 0.8 and up
// 15-18 % slower; after one or two full rounds, up to 0.22 16-23 %, 0.27-0.48
// 2-8 % faster, 0.6 8-13 % slower; after three or more, 0.05-0.22 8-15 % faster, 0.36 1-2 %
// slower.  FP32: 2.4x, 1.5x; 1.16-1.46x, 1.07-1.11x; 1.03-1.16x.  From 16
// rounds on the remainder is noise.
int gram_full_tiles(int n_tiles, int quads, int n_cu)
{
    const int rem = n_tiles % n_cu, rounds = n_tiles / n_cu;
    const int most = rounds < 3 ? 2 * n_cu : n_cu;  // 32 x 32 tiles, one or two per CU
    return rounds < 16 && quads * rem <= most ? n_tiles - rem : n_tiles;
}

void launch_gram(const GramArgs& a, GramMode mode, hipStream_t s)
{
    if (a.n_tiles <= 0) return;
    const int n_quad = a.quads * (a.n_tiles - a.n_full);
    const int grid = ((a.n_full + kXcd - 1) / kXcd + (n_quad + kXcd - 1) / kXcd) * kXcd;
    const bool st = a.stats_part != nullptr;
    if (mode == kGramBF16x3 && st)
        gram_kernel<kGramBF16x3, true><<<grid, 256, 0, s>>>(a);
    else if (mode == kGramBF16x3)
        gram_kernel<kGramBF16x3, false><<<grid, 256, 0, s>>>(a);
    else if (st)
        gram_kernel<kGramFP32, true><<<grid, 256, 0, s>>>(a);
    else
        gram_kernel<kGramFP32, false><<<grid, 256, 0, s>>>(a);
}

void launch_zero_u32(uint32_t* p, int n, hipStream_t s)
{
    zero_u32_kernel<<<(n + 255) / 256, 256, 0, s>>>(p, n);
}

void launch_zero_words(uint32_t* p, int64_t n_words, hipStream_t s)
{
    // callers allocate bitmaps in whole 16-byte units
    const int64_t n4 = (n_words + 3) / 4;
    const int64_t blocks = std::min<int64_t>(4096, std::max<int64_t>(1, (n4 + 255) / 256));
    zero_words_kernel<<<(int)blocks, 256, 0, s>>>(reinterpret_cast<uint4*>(p), n4);
}

void launch_flag_resolve(const double* xyz_a, const double* cent_a, const double* xyz_b,
                         const double* cent_b, int L, uint32_t* ctl, const int64_t* list, int cap,
                         uint32_t* bits, int64_t n_out, int triangle, int n, int64_t out_ld, void* out,
                         int out_f64, uint32_t* h_report, unsigned* st_min, unsigned* st_max,
                         uint64_t* clk, bool ends_call, hipStream_t s)
{
    // 1024 waves: a typical list (tens to thousands of pairs) is one trip of a
    // few pairs per wave.  Short chains flag up to half of their pairs and
    // get twice as many where there is enough to do (2000 x 20 370 -> 299 us,
    // 6000 x 60 84 -> 58; four times as many: 264 and 55, but 22 instead of 15
    // for 2000 x 60).
    const int groups = L <= kShortChain && n_out >= (int64_t)1 << 19 ? 512 : 256;
    static_assert(256 % kFlagLists == 0, "every list has the same number of groups");
    flag_resolve_kernel<<<groups, 64 * kResolveWaves, 0, s>>>(
        xyz_a, cent_a, xyz_b, cent_b, L, ctl, list, cap, bits, n_out, triangle, n, out_ld, out, out_f64,
        h_report, st_min, st_max, clk, ends_call ? 1 : 0);
}

void launch_flag_compact(uint32_t* bits, int64_t n_words, int64_t* list, int cap, uint32_t* count,
                         hipStream_t s)
{
    const int64_t blocks = std::min<int64_t>(4096, std::max<int64_t>(1, (n_words + 255) / 256));
    flag_compact_kernel<<<(int)blocks, 256, 0, s>>>(bits, n_words, list, cap, count);
}

}  // namespace bs
