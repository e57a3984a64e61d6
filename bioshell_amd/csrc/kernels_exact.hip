// kernels_exact.hip -- all-vs-all cRMSD in FP64 (BS_FP64_PLAIN): the textbook
// steps of every pair (centroid = sum / n, subtract, 3x3 cross-covariance of
// the centred sets, QCP from E0, RMSD) with the covariance on the FP64 matrix
// unit.  v_mfma_f64_16x16x4_f64 rounds each multiply-add like a v_fma_f64 and
// runs at the same rate; what it saves is the operands: nine 16 x 16 tiles of
// covariances share three row and three column values per lane, where a
// thread of the per-pair kernel fetched 6 values from LDS for 36 multiply-adds
// and was bound by that (kernels_plain.hip: the LDS's 128 bytes a clock).
//
// Accumulator slot r of lane l holds row 4 r + l / 16, column l % 16.
#include <algorithm>

#include "common.hpp"
#include "exact_solve.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace bs {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x2a8 __attribute__((ext_vector_type(2), aligned(8)));  // two doubles, 8-byte aligned

__device__ inline int64_t tri_index(int64_t n, int64_t i, int64_t j)
{
    return i * n - i * (i + 1) / 2 + (j - i - 1);
}

// Linear block id -> (bi, bj), bi <= bj, over an nt x nt upper triangle.
__device__ inline void tri_tile(int64_t b, int nt, int& bi, int& bj)
{
    const double twon1 = 2.0 * nt + 1.0;
    int r = (int)floor((twon1 - sqrt(twon1 * twon1 - 8.0 * (double)b)) * 0.5);
    auto start = [nt](int64_t row) { return row * nt - row * (row - 1) / 2; };
    while (r > 0 && start(r) > b) --r;
    while (start(r + 1) <= b) ++r;
    bi = r;
    bj = r + (int)(b - start(r));
}

__device__ inline void mfma9(const double (&a)[3], const double (&b)[3], f64x4 (&acc)[9])
{
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d)
            acc[3 * c + d] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[c], b[d], acc[3 * c + d], 0, 0, 0);
}

__device__ inline void store_pair(void* __restrict__ out, int out_f64, int n, int i, int j, double r)
{
    const int64_t o = tri_index(n, i, j);
    if (out_f64)
        static_cast<double*>(out)[o] = r;
    else
        static_cast<float*>(out)[o] = (float)r;
}

// ------------------------------------------------------------ small ensembles
// One work-group per 16 x 16 pairs, in one launch: the tile's 32 conformations
// are read into LDS once, centred there, the atoms are dealt to the four waves
// four at a time, and after the waves' partial covariances are added every
// thread solves one pair.  Bound: latency, one round of work-groups (200 x 76, in
// us: reads 2.2, centroids 1.6, products 2.0, sums 0.5, solve 1.4).  200 x 76
// takes 9.0 us, the per-pair kernel 16.5; one pair 8.0 and 12.
constexpr int kExactThreads = 256;

__global__ __launch_bounds__(kExactThreads, 2) void exact_small_kernel(const double* __restrict__ xyz, int n, int L,
                                                                    int nt, void* __restrict__ out, int out_f64,
                                                                    uint64_t* t_start, uint64_t* t_end)
{
    // sized by the launch (exact_small_lds): with a static array the compiler
    // sees one wave per SIMD and copies the accumulators between its two register
    // files around every step
    extern __shared__ __align__(16) double lds[];
    double(*cen)[4] = reinterpret_cast<double(*)[4]>(lds);  // centroid, sum of squares of the 32 conformations
    double* sm = lds + 32 * 4;
    stamp_start(t_start);
    int bi, bj;
    tri_tile(blockIdx.x, nt, bi, bj);
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int ld = (3 * L) | 1;  // odd: consecutive conformations start in different banks
    {
        // conformations w, w + 4, ...: 16 bytes a lane, eight conformations in flight
        const double* src[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = w + 4 * u;
            const int conf = min(c < 16 ? bi * 16 + c : bj * 16 + (c - 16), n - 1);
            src[u] = xyz + (int64_t)conf * L * 3;
        }
#pragma unroll 2
        for (int v = 2 * lane; v < 3 * L; v += 128) {
            f64x2a8 x[8];
            const bool both = v + 1 < 3 * L;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (both) {
                    x[u] = *reinterpret_cast<const f64x2a8*>(src[u] + v);
                } else {
                    x[u][0] = src[u][v];
                    x[u][1] = 0.0;
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                sm[(w + 4 * u) * ld + v] = x[u][0];
                if (both) sm[(w + 4 * u) * ld + v + 1] = x[u][1];
            }
        }
    }
    __syncthreads();
    {
        const int c = t >> 3, part = t & 7;
        const double* p = sm + c * ld;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, g = 0.0;
#pragma unroll 4
        for (int k = part; k < L; k += 8) {
            s0 += p[3 * k];
            s1 += p[3 * k + 1];
            s2 += p[3 * k + 2];
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            s0 += __shfl_xor(s0, o);
            s1 += __shfl_xor(s1, o);
            s2 += __shfl_xor(s2, o);
        }
        s0 /= L;
        s1 /= L;
        s2 /= L;
#pragma unroll 4
        for (int k = part; k < L; k += 8) {
            const double x = p[3 * k] - s0, y = p[3 * k + 1] - s1, z = p[3 * k + 2] - s2;
            g += x * x + y * y + z * z;
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) g += __shfl_xor(g, o);
        if (part < 4) cen[c][part] = part == 0 ? s0 : part == 1 ? s1 : part == 2 ? s2 : g;
    }
    __syncthreads();
    const int row = lane & 15, grp = lane >> 4;
    f64x4 acc[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
    {
        const double* pa = sm + row * ld;
        const double* pb = sm + (16 + row) * ld;
        double ca[3], cb[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            ca[c] = cen[row][c];
            cb[c] = cen[16 + row][c];
        }
        for (int k = 4 * w + grp; k - grp < L; k += 16) {  // uniform trip count per wave
            double a[3], b[3];
            const int kk = k < L ? k : 0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {  // read unconditionally: no branch around the reads
                a[c] = pa[3 * kk + c] - ca[c];
                b[c] = pb[3 * kk + c] - cb[c];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                a[c] = k < L ? a[c] : 0.0;
                b[c] = k < L ? b[c] : 0.0;
            }
            mfma9(a, b, acc);
        }
    }
    __syncthreads();  // the coordinates' LDS takes the partial covariances
#pragma unroll
    for (int q = 0; q < 9; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) sm[(w * 9 + q) * 256 + (4 * r + grp) * 16 + row] = acc[q][r];
    __syncthreads();
    const int i = bi * 16 + (t >> 4), j = bj * 16 + (t & 15);
    if (i < j && j < n) {
        double m[9];
#pragma unroll
        for (int q = 0; q < 9; ++q)
            m[q] = (sm[q * 256 + t] + sm[(9 + q) * 256 + t]) + (sm[(18 + q) * 256 + t] + sm[(27 + q) * 256 + t]);
        store_pair(out, out_f64, n, i, j, exact_rmsd(m, cen[t >> 4][3], cen[16 + (t & 15)][3], L));
    }
    stamp_end(t_end);
}

// ------------------------------------------------------------ the rest
// Centroid and sum of squares about it, one wave per conformation.
__global__ __launch_bounds__(256) void exact_centre_kernel(const double* __restrict__ xyz, int n, int L,
                                                           double* __restrict__ cg, uint64_t* t_start)
{
    stamp_start(t_start);
    const int conf = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (conf >= n) return;
    const double* p = xyz + (int64_t)conf * L * 3;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, g = 0.0;
#pragma unroll 4
    for (int k = lane; k < L; k += 64) {
        s0 += p[3 * k];
        s1 += p[3 * k + 1];
        s2 += p[3 * k + 2];
    }
    s0 = wave_sum(s0) / L;
    s1 = wave_sum(s1) / L;
    s2 = wave_sum(s2) / L;
#pragma unroll 4
    for (int k = lane; k < L; k += 64) {
        const double x = p[3 * k] - s0, y = p[3 * k + 1] - s1, z = p[3 * k + 2] - s2;
        g += x * x + y * y + z * z;
    }
    g = wave_sum(g);
    if (lane < 4) cg[4 * (int64_t)conf + lane] = lane == 0 ? s0 : lane == 1 ? s1 : lane == 2 ? s2 : g;
}

// One work-group per 32 x 32 pairs, wave w the 16 x 16 block (w / 2, w % 2).
// The tile's 64 conformations stream through LDS in chunks of 8 atoms, two
// buffers, centred on the way.  Each lane then solves its four pairs.  LDS row
// 3 (atom / 2) + coordinate holds two atoms' values per conformation, 16 bytes
// that a lane reads at once for two steps of products (atoms 2 l/16 and
// 2 l/16 + 1); within a row the conformations are permuted by the row's number,
// so that the rows a store writes for one conformation fall into different
// banks, and 16 lanes of a load still read 256 contiguous bytes.
//
// Bound: the FP64 matrix unit, 58 % busy at 1501 x 600 (0.29 ms, 42 TFLOP/s; a
// large FP64 product reaches 69), with 4.4 tiles per CU of which some get 5.
// FP64 additions hold the unit up: centring as the values are staged (6 per
// thread and chunk) instead of as each wave reads its operands (12) took 0.31 to
// 0.29 ms.  1501 x 211: 124 us, the per-pair kernel's 261; 3000 x 100: 235 and
// 436.  A second chunk in flight at two work-groups per CU, and rows padded
// instead of permuted, changed nothing.
constexpr int kExactChunk = 8;
__device__ inline int exact_pos(int row, int c) { return (row * 64 + (c ^ row)) * 2; }

__global__ __launch_bounds__(kExactThreads, 3) void exact_tile_kernel(const double* __restrict__ xyz, int n, int L,
                                                                      int nt, const double* __restrict__ cg,
                                                                      void* __restrict__ out, int out_f64,
                                                                      uint64_t* t_end)
{
    __shared__ __align__(16) double buf[2][kExactChunk * 3 * 64];
    int bi, bj;
    tri_tile(blockIdx.x, nt, bi, bj);
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wr = w >> 1, wc = w & 1, row = lane & 15, grp = lane >> 4;
    constexpr int kParts = kExactChunk * 3 / 2, kPer = 64 * kParts / kExactThreads;  // pairs of doubles
    static_assert(64 * kParts % kExactThreads == 0, "staging shape");
    const double* src[kPer];
    int part[kPer], dst0[kPer], dst1[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int e = t + kExactThreads * u, c = e / kParts;
        part[u] = 2 * (e - c * kParts);
        const int conf = min(c < 32 ? bi * 32 + c : bj * 32 + (c - 32), n - 1);
        src[u] = xyz + (int64_t)conf * L * 3 + part[u];
        auto pos = [c](int e) { return exact_pos(e / 6 * 3 + e % 3, c) + (e / 3 & 1); };
        dst0[u] = pos(part[u]);
        dst1[u] = pos(part[u] + 1);
    }
    double c0[kPer], c1[kPer];  // the values' centroid coordinates
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int e = t + kExactThreads * u, c = e / kParts;
        const double* cc = cg + 4 * (int64_t)min(c < 32 ? bi * 32 + c : bj * 32 + (c - 32), n - 1);
        c0[u] = cc[part[u] % 3];
        c1[u] = cc[(part[u] + 1) % 3];
    }
    f64x2a8 x[kPer];
    auto load = [&](int k0) {
        if (k0 + kExactChunk <= L) {  // uniform
#pragma unroll
            for (int u = 0; u < kPer; ++u) x[u] = *reinterpret_cast<const f64x2a8*>(src[u] + 3 * (int64_t)k0);
        } else {  // the atoms past the chain's end: their centroid, 0 once centred
            const int left = 3 * (L - k0);
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const double* p = src[u] + (3 * (int64_t)k0 - part[u]);
                const double y0 = p[min(part[u], left - 1)], y1 = p[min(part[u] + 1, left - 1)];
                x[u] = f64x2a8{part[u] < left ? y0 : c0[u], part[u] + 1 < left ? y1 : c1[u]};
            }
        }
    };
    auto store = [&](double* to) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            to[dst0[u]] = x[u][0] - c0[u];
            to[dst1[u]] = x[u][1] - c1[u];
        }
    };
    const int jb = min(bj * 32 + wc * 16 + row, n - 1);
    int ra[3], rb[3];  // this lane's operands in a buffer
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        ra[c] = exact_pos(3 * grp + c, wr * 16 + row);
        rb[c] = exact_pos(3 * grp + c, 32 + wc * 16 + row);
    }
    const bool active = bi < bj || wr <= wc;  // else every pair of the wave is below the diagonal
    f64x4 acc[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
    load(0);
    store(buf[0]);
    __syncthreads();
    for (int k0 = 0, b = 0; k0 < L; k0 += kExactChunk, b ^= 1) {
        const bool more = k0 + kExactChunk < L;
        if (more) load(k0 + kExactChunk);
        if (active) {
            f64x2 a2[3], b2[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                a2[c] = *reinterpret_cast<const f64x2*>(&buf[b][ra[c]]);
                b2[c] = *reinterpret_cast<const f64x2*>(&buf[b][rb[c]]);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const double av[3] = {a2[0][s], a2[1][s], a2[2][s]}, bv[3] = {b2[0][s], b2[1][s], b2[2][s]};
                mfma9(av, bv, acc);
            }
        }
        if (more) store(buf[b ^ 1]);
        __syncthreads();
    }
    const int j = bj * 32 + wc * 16 + row;
    const double gj = cg[4 * (int64_t)jb + 3];
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
        const int i = bi * 32 + wr * 16 + 4 * r + grp;
        if (i >= j || j >= n) continue;
        double m[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) m[q] = r == 0 ? acc[q][0] : r == 1 ? acc[q][1] : r == 2 ? acc[q][2] : acc[q][3];
        store_pair(out, out_f64, n, i, j, exact_rmsd(m, cg[4 * (int64_t)i + 3], gj, L));
    }
    stamp_end(t_end, kStampUniform);
}

constexpr int kLdsBytes = 160 * 1024;

// The small kernel's LDS: the tile's coordinates, later the waves' covariances.
size_t exact_small_lds(int L)
{
    return (32 * 4 + std::max<size_t>(32 * ((3 * (size_t)L) | 1), 4 * 9 * 256)) * 8;
}

// ------------------------------------------------------------------ one pair
// Two conformations of at most 256 kPairAtoms atoms by one work-group, every
// atom in registers, read once: a and b, like the result, may be pinned host
// memory, which the copies to and from the device cost more than the reads
// over the bus do.  Bound by latency: a call for 76 atoms takes 20 us, 39 with
// two copies in, the tile kernel and a copy out.
constexpr int kPairAtoms = kPairMaxAtoms / 256;

template <int N>
__device__ inline void pair_sum(double (&v)[N], double (*part)[11])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = wave_sum(v[q]);
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < N; ++q) part[w][q] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = (part[0][q] + part[1][q]) + (part[2][q] + part[3][q]);
    __syncthreads();
}

__global__ __launch_bounds__(256) void pair_kernel(const double* a, const double* b, int L, double* out,
                                                   uint64_t* t_start, uint64_t* t_end)
{
    __shared__ double part[4][11];
    stamp_start(t_start);
    double x[kPairAtoms][6];
    double c[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < kPairAtoms; ++j) {
        if (256 * j >= L) break;  // uniform
        const int k = 3 * min((int)threadIdx.x + 256 * j, L - 1);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            x[j][q] = a[k + q];
            x[j][3 + q] = b[k + q];
        }
    }
#pragma unroll
    for (int j = 0; j < kPairAtoms; ++j) {
        if (256 * j >= L) break;
        const bool in = (int)threadIdx.x + 256 * j < L;
#pragma unroll
        for (int q = 0; q < 6; ++q) c[q] += in ? x[j][q] : 0.0;
    }
    pair_sum<6>(c, part);
    double v[11] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};  // covariance, inner products
#pragma unroll
    for (int j = 0; j < kPairAtoms; ++j) {
        if (256 * j >= L) break;
        const bool in = (int)threadIdx.x + 256 * j < L;
        double d[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) d[q] = in ? x[j][q] - c[q] / L : 0.0;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int q = 0; q < 3; ++q) v[3 * p + q] += d[p] * d[3 + q];
            v[9] += d[p] * d[p];
            v[10] += d[3 + p] * d[3 + p];
        }
    }
    pair_sum<11>(v, part);
    if (threadIdx.x < 64) {
        const double m[9] = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8]};
        const double r = exact_rmsd(m, v[9], v[10], L);
        if (threadIdx.x == 0) {
            *out = r;
            if (t_end) *t_end = wall_clock64();
        }
    }
}

}  // namespace

void launch_pair(const double* a, const double* b, int L, double* out, hipStream_t s, uint64_t* clk)
{
    pair_kernel<<<1, 256, 0, s>>>(a, b, L, out, clk ? clk + kClkStart : nullptr, clk ? clk + kClkEnds : nullptr);
}

// One launch while the LDS holds the coordinates (up to 211 atoms) and every
// work-group is resident at once: a second round costs more than the second
// launch and the staged reads save (us, one launch against two: 300 x 76 10.4
// and 19.0, 400 x 76 12.8 and 19.2, 500 x 76 21.9 and 20.0; 300 x 200 15.7 and
// 31.4, 500 x 150 38.9 and 27.7).
bool exact_small(int n, int L, int n_cu)
{
    const int64_t nt = (n + 15) / 16;
    const size_t lds = exact_small_lds(L);
    return lds <= kLdsBytes && nt * (nt + 1) / 2 <= (int64_t)(kLdsBytes / lds) * n_cu;
}

// The limit is the kernel's, for every thread and context: set once to the
// most any launch asks for, never to the size of one of them, which another
// thread's launch may already exceed.
void exact_init()
{
    BS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&exact_small_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));
}

size_t exact_scratch_bytes(int n, int L, int n_cu) { return exact_small(n, L, n_cu) ? 0 : (size_t)n * 32; }

void launch_exact_avsa(const double* xyz, int n, int L, void* out, bool out_f64, int n_cu, double* scratch,
                       hipStream_t s, uint64_t* clk)
{
    if (n < 2) return;
    uint64_t *t0 = clk ? clk + kClkStart : nullptr, *t1 = clk ? clk + kClkEnds : nullptr;
    const int f = out_f64 ? 1 : 0;
    if (exact_small(n, L, n_cu)) {
        const int nt = (n + 15) / 16, grid = nt * (nt + 1) / 2;
        const int lds = (int)exact_small_lds(L);
        exact_small_kernel<<<grid, kExactThreads, lds, s>>>(xyz, n, L, nt, out, f, t0, t1);
        return;
    }
    const int nt = (n + 31) / 32;
    exact_centre_kernel<<<(n + 3) / 4, 256, 0, s>>>(xyz, n, L, scratch, t0);
    exact_tile_kernel<<<(unsigned)((int64_t)nt * (nt + 1) / 2), kExactThreads, 0, s>>>(xyz, n, L, nt, scratch, out, f,
                                                                                        t1);
}

}  // namespace bs
