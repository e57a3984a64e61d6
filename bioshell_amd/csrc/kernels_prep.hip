// kernels_prep.hip -- single-ensemble launches of the preparation steps
// (bodies and the data flow in prep_device.hpp) and the single-pair
// superposition kernel.
#include "prep_device.hpp"

namespace bs {
namespace {

// Fit + pack forms the reference itself for at most this many atoms (what fits
// in LDS beside the rest with three groups on a CU) and slices of samples (32:
// up to 4100 conformations; every group reads them all, and the gain is down
// to 1.3 us at 24).
constexpr int kFoldAtoms = 832;
constexpr int kFoldSlices = 32;

bool folds_mean(int S, int L) { return L <= kFoldAtoms && ref_slices(S) <= kFoldSlices; }

// Reference: the fits of the S samples onto conformation 0 and their
// rotated sums, one slice of samples per work-group (fit0_slice),
// the mean (thread per coordinate, one wave per work-group to spread the few
// coordinates over more CUs), then R0 (one block).
__global__ __launch_bounds__(256) void fit0_kernel(const double* __restrict__ xyz, int n, int S,
                                                   int L, double* __restrict__ partial, uint64_t* t_start)
{
    __shared__ Fit0Lds lds;
    stamp_start(t_start);
    fit0_slice(xyz, n, S, L, blockIdx.x, partial, lds);
}

__global__ __launch_bounds__(64) void mean_final_kernel(const double* __restrict__ partial,
                                                         int n_slices, int S, int L,
                                                         double* __restrict__ ref)
{
    const int v = blockIdx.x * 64 + threadIdx.x;
    if (v >= 3 * L) return;
    mean_final_coord(partial, n_slices, S, L, v, ref);
}

__global__ __launch_bounds__(256) void ref_gram_kernel(double* __restrict__ ref, int L)
{
    __shared__ double part[4][6];
    ref_gram_block(ref, L, part);
}

// MEAN: the reference is formed here, by every work-group for itself from the
// fitted samples' partial sums (in LDS; the first group also writes it to ref,
// with R0).  Bound by latency, like the two launches of 4.6 us it replaces:
// preparation of 2000 x 150 32.8 -> 30.7 us, 500 x 120 26.2 -> 23.6, 3001 x 187
// (24 slices) 35.5 -> 34.2.
template <int MODE, bool MEAN>
__global__ __launch_bounds__(256) void fit_pack_kernel(const double* __restrict__ xyz, double* __restrict__ ref,
                                                       const double* __restrict__ partial, int n_slices, int S,
                                                       int n, int n_pad, int L, int n_kblk,
                                                       double* __restrict__ rot,
                                                       double* __restrict__ cent,
                                                       uint4* __restrict__ panels,
                                                       double* __restrict__ consts, int ld,
                                                       uint64_t* t_start)
{
    __shared__ FitPackLds lds;
    stamp_start(t_start);
    const int blk = xcd_contiguous_block(fit_groups(n_pad));
    if (blk < 0) return;
    if constexpr (MEAN) {
        __shared__ double r[3 * kFoldAtoms + 6];
        __shared__ double part[4][6];
        for (int v = threadIdx.x; v < 3 * L; v += 256)
            r[v] = n_slices <= 16 ? mean_few_slices<16>(partial, n_slices, S, L, v)
                                  : mean_few_slices<kFoldSlices>(partial, n_slices, S, L, v);
        __syncthreads();
        ref_gram_block(r, L, part);
        __syncthreads();
        if (blk == 0)
            for (int v = threadIdx.x; v < 3 * L + 6; v += 256) ref[v] = r[v];
        fit_pack_block<MODE>(xyz, r, n, L, n_kblk, blk * kFitConfs, rot, cent, panels, consts, ld, lds);
        return;
    }
    fit_pack_block<MODE>(xyz, ref, n, L, n_kblk, blk * kFitConfs, rot, cent, panels, consts, ld, lds);
}

// ------------------------------------------------------ single superposition
__global__ __launch_bounds__(64) void superpose_kernel(const double* __restrict__ a,
                                                       const double* __restrict__ b, int L,
                                                       double* __restrict__ out)
{
    const int lane = threadIdx.x;
    double sa[3] = {0, 0, 0}, sb[3] = {0, 0, 0};
    for (int k = lane; k < L; k += 64)
        for (int c = 0; c < 3; ++c) {
            sa[c] += a[3 * k + c];
            sb[c] += b[3 * k + c];
        }
    for (int c = 0; c < 3; ++c) {
        sa[c] = wave_sum(sa[c]) / L;
        sb[c] = wave_sum(sb[c]) / L;
    }
    double m[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    double ga = 0, gb = 0;
    for (int k = lane; k < L; k += 64) {
        double pa[3], pb[3];
        for (int c = 0; c < 3; ++c) {
            pa[c] = a[3 * k + c] - sa[c];
            pb[c] = b[3 * k + c] - sb[c];
        }
        for (int p = 0; p < 3; ++p)
            for (int q = 0; q < 3; ++q) m[3 * p + q] += pb[p] * pa[q];
        ga += pa[0] * pa[0] + pa[1] * pa[1] + pa[2] * pa[2];
        gb += pb[0] * pb[0] + pb[1] * pb[1] + pb[2] * pb[2];
    }
    for (int q = 0; q < 9; ++q) m[q] = wave_sum(m[q]);
    ga = wave_sum(ga);
    gb = wave_sum(gb);
    if (lane == 0) {
        double R[9], lam;
        rotation_from_cov(m, R, &lam);
        for (int q = 0; q < 9; ++q) out[q] = R[q];
        for (int r = 0; r < 3; ++r)
            out[9 + r] = sa[r] - (R[3 * r] * sb[0] + R[3 * r + 1] * sb[1] + R[3 * r + 2] * sb[2]);
        const double r2 = 2.0 * (0.5 * (ga + gb) - lam) / L;
        out[12] = sqrt(r2 > 0.0 ? r2 : 0.0);
    }
}

__global__ __launch_bounds__(256) void copy_doubles_kernel(double* __restrict__ dst, const double* __restrict__ src,
                                                           int64_t n)
{
    const int64_t v = 2 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (v + 1 < n)
        *reinterpret_cast<double2*>(dst + v) = *reinterpret_cast<const double2*>(src + v);
    else if (v < n)
        dst[v] = src[v];
}

}  // namespace

void launch_copy_doubles(double* dst, const double* src, int64_t n, hipStream_t s)
{
    copy_doubles_kernel<<<(unsigned)((n + 511) / 512), 256, 0, s>>>(dst, src, n);
}

void launch_prepare(const double* xyz, int n, int L, int n_pad, int n_kblk, GramMode mode, const double* fixed_ref,
                    double* partial, double* ref, double* rot, double* cent, void* panels, double* consts, int ld,
                    hipStream_t s, uint64_t* t_start)
{
    const int S = ref_sample_count(n), slices = ref_slices(S);
    const bool fold = !fixed_ref && folds_mean(S, L);
    if (!fixed_ref) {
        fit0_kernel<<<slices, 256, 0, s>>>(xyz, n, S, L, partial, t_start);
        t_start = nullptr;
        if (!fold) {
            mean_final_kernel<<<(3 * L + 63) / 64, 64, 0, s>>>(partial, slices, S, L, ref);
            ref_gram_kernel<<<1, 256, 0, s>>>(ref, L);
        }
    }
    double* r = fixed_ref ? const_cast<double*>(fixed_ref) : ref;  // written only where folded
    const int blocks = xcd_contiguous_grid(fit_groups(n_pad));
    uint4* p = static_cast<uint4*>(panels);
#define BS_FIT_PACK(M, FOLD)                                                                                     \
    fit_pack_kernel<M, FOLD><<<blocks, 256, 0, s>>>(xyz, r, partial, slices, S, n, n_pad, L, n_kblk, rot, cent, p, \
                                                    consts, ld, t_start)
    if (mode == kGramBF16x3) {
        if (fold)
            BS_FIT_PACK(kGramBF16x3, true);
        else
            BS_FIT_PACK(kGramBF16x3, false);
    } else {
        if (fold)
            BS_FIT_PACK(kGramFP32, true);
        else
            BS_FIT_PACK(kGramFP32, false);
    }
#undef BS_FIT_PACK
}

void launch_superpose(const double* a, const double* b, int L, double* out13, hipStream_t s)
{
    superpose_kernel<<<1, 64, 0, s>>>(a, b, L, out13);
}

}  // namespace bs
