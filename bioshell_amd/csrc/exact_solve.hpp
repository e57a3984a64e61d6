// exact_solve.hpp -- the FP64 QCP solve of the exact kernels and of the
// re-evaluation of flagged pairs.
#pragma once

#include "qcp.hpp"

namespace bs {

// The near-degenerate polish of the QCP solve, taken by few pairs if any: out
// of line, so that its 4 x 4 matrices do not cost every pair registers.
static __device__ __attribute__((noinline)) double exact_polish(double m0, double m1, double m2, double m3, double m4,
                                                         double m5, double m6, double m7, double m8)
{
    const double m[9] = {m0, m1, m2, m3, m4, m5, m6, m7, m8};
    return qcp_polish<double>(m);
}

// qcp_rmsd (qcp.hpp) with two changes to the Newton iteration.  It starts from
// the smaller of E0 and
//     (|M|^2 + 2 sqrt(3 sum of the squared 2 x 2 minors))^(1/2) >= s1 + s2 + s3 >= lambda,
// s the singular values (the sum of their products is at most sqrt(3) times the
// root of the sum of the products' squares), which for pairs that fit badly is
// far nearer: 3 to 4 steps instead of 6 to 10, and no pair is polished only
// for its number of steps.  And the step's quotient is rcp with two refinements.
// A lane that is not live (its sums are zeros, which would ask for the polish)
// returns anything.
__device__ inline double exact_rmsd(const double (&m)[9], double gi, double gj, int L, bool live = true)
{
    double f2 = 0.0;
#pragma unroll
    for (int q = 0; q < 9; ++q) f2 += m[q] * m[q];
    double minors = 0.0;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int a = (p + 1) % 3, b = (p + 2) % 3, c = (q + 1) % 3, d = (q + 2) % 3;
            const double v = m[3 * a + c] * m[3 * b + d] - m[3 * a + d] * m[3 * b + c];
            minors += v * v;
        }
    const double c2 = -2.0 * f2, c1 = -8.0 * det3(m), c0 = det_key(m);
    const double E0 = 0.5 * (gi + gj);
    double l = fmin(E0, sqrt(f2 + 2.0 * sqrt(3.0 * minors)) * (1.0 + 4e-15)), dp = 0.0;
    int it = 0;
    while (it < 50) {
        const double l2 = l * l;
        const double p = ((l2 + c2) * l + c1) * l + c0;
        dp = (4.0 * l2 + 2.0 * c2) * l + c1;
        if (dp == 0.0) break;
        const double step = newton_div(p, dp);
        l -= step;
        ++it;
        if (fabs(step) <= 1e-11 * fabs(l)) break;
    }
    const double scale = fabs(4.0 * l * l * l) + fabs(2.0 * c2 * l) + fabs(c1);
    if (live & ((it > 8) | !(fabs(dp) > 1e-4 * scale))) l = exact_polish(m[0], m[1], m[2], m[3], m[4], m[5], m[6], m[7], m[8]);
    const double r2 = 2.0 * (E0 - l) / L;
    return sqrt(r2 > 0.0 ? r2 : 0.0);
}

}  // namespace bs
