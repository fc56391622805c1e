// rf_inner.h -- device math shared by the assembly kernel and the
// matrix-free operator: the Legendre monomial coefficients and the analytic
// moments I, J, S of the inner integral (fortran/Int_analytical.f90:5-293).
#pragma once

#include "rf_internal.h"

#include <type_traits>

namespace rf {
namespace {

// Coefficients of P_l(s) = sum_m c[l][m] s^m (the combinations of
// fortran/Int_analytical.f90:213-288).
__device__ constexpr double kLeg[9][9] = {
    {1, 0, 0, 0, 0, 0, 0, 0, 0},
    {0, 1, 0, 0, 0, 0, 0, 0, 0},
    {-0.5, 0, 1.5, 0, 0, 0, 0, 0, 0},
    {0, -1.5, 0, 2.5, 0, 0, 0, 0, 0},
    {0.375, 0, -3.75, 0, 4.375, 0, 0, 0, 0},
    {0, 1.875, 0, -8.75, 0, 7.875, 0, 0, 0},
    {-0.3125, 0, 6.5625, 0, -19.6875, 0, 14.4375, 0, 0},
    {0, -2.1875, 0, 19.6875, 0, -43.3125, 0, 26.8125, 0},
    {0.2734375, 0, -9.84375, 0, 54.140625, 0, -93.84375, 0, 50.2734375},
};

// Symmetric 3x3 <-> 6-vector (11,22,33,12,13,23).
__device__ __forceinline__ int sym6(int a, int b)
{
    return (a == b) ? a : (a + b + 2);  // (0,1)->3 (0,2)->4 (1,2)->5
}

// Moments of the analytic inner integral at point X against fiber (xj,tj):
// I_n, J_n, S_n = integral over s in [-1,1] of s^n / |R|^{1,3,5}, n = 0..M+2,
// R = X - xj - s tj (fortran/Int_analytical.f90:5-207).  The closed forms of
// n = 0, 1 (logarithms, square roots, the 1/d terms) and the forward
// recurrences of the near field (c < 10) are FP64; RB is the arithmetic type
// of the 26-step backward recurrences of the far field (double, or float in
// mixed precision, whose error is then ~FP32 rounding of the moments).
// BRANCH: the recurrences by c (kByDistance), or those the caller knows to apply.
// YFIRST: which product of the three-term sums b and c is rounded first.  Near
// a source's axis line and for |R|^2 around 10 the closed forms and recurrences
// amplify their last bit up to 1e-6 of an entry, so the order is written out
// and not left to the compiler's choice of fused operations.
enum MomentBranch { kByDistance, kForward, kBackward };
template <int M>
struct Moments {
    double r0x, r0y, r0z, px, py, pz;
    double I[M + 3], J[M + 3], S[M + 3];
};

template <int M, typename RB, MomentBranch BRANCH = kByDistance, bool YFIRST = false>
__device__ __forceinline__ void analytic_moments(double X0, double X1, double X2, const double* xj, const double* tj,
                                                 Moments<M>& mo)
{
    constexpr int NM = M + 3;  // moments 0..M+2
    const double r0x = X0 - xj[0], r0y = X1 - xj[1], r0z = X2 - xj[2];
    const double px = tj[0], py = tj[1], pz = tj[2];
    const double b = -2.0 * fma(pz, r0z, YFIRST ? fma(py, r0y, px * r0x) : fma(px, r0x, py * r0y));
    const double c = fma(r0z, r0z, YFIRST ? fma(r0y, r0y, r0x * r0x) : fma(r0x, r0x, r0y * r0y));
    const double ue = sqrt(1.0 + b + c);
    const double ub = sqrt(1.0 - b + c);
    const double d = c - 0.25 * b * b;
    double* I = mo.I;
    double* J = mo.J;
    double* S = mo.S;
    I[0] = log(fabs(2.0 + b + 2.0 * ue)) - log(fabs(-2.0 + b + 2.0 * ub));
    I[1] = ue - ub - 0.5 * b * I[0];
    const double iue = 1.0 / ue, iub = 1.0 / ub;
    if (d < 1e-14) {  // collinear (Int_analytical.f90:162-169,189-196)
        const double sp = 1.0 + 0.5 * b, sm = -1.0 + 0.5 * b;
        J[0] = -0.5 / (sp * sp) + 0.5 / (sm * sm);
        J[1] = -iue + iub - 0.5 * b * J[0];
        const double ap = 2.0 + b, am = -2.0 + b;
        S[0] = -4.0 / (ap * ap * ap * ap) + 4.0 / (am * am * am * am);
        S[1] = -8.0 / (3.0 * ap * ap * ap) + 8.0 / (3.0 * am * am * am) - 0.5 * b * S[0];
    } else {
        const double id = 1.0 / d;
        J[0] = ((1.0 + 0.5 * b) * iue - (-1.0 + 0.5 * b) * iub) * id;
        J[1] = -iue + iub - 0.5 * b * J[0];
        const double iue3 = iue * iue * iue, iub3 = iub * iub * iub;
        const double i6d = id * (1.0 / 6.0);
        S[0] = ((2.0 + b) * iue3 - (-2.0 + b) * iub3) * i6d + ((2.0 / 3.0) * id) * J[0];
        S[1] = (-(b + 2.0 * c) * iue3 + (2.0 * c - b) * iub3) * i6d - (b * id * (1.0 / 3.0)) * J[0];
    }
    if (BRANCH == kForward || (BRANCH == kByDistance && c < 10.0)) {
        // forward recurrences (Int_analytical.f90:123-136,172-176,197-200)
#pragma unroll
        for (int n = 2; n < NM; ++n) {
            const double sgn = (n % 2 == 1) ? 1.0 : -1.0;  // (-1)^(n-1)
            I[n] = (ue - sgn * ub) * (1.0 / n) - ((n - 0.5) / n) * b * I[n - 1] - ((n - 1.0) / n) * c * I[n - 2];
            J[n] = I[n - 2] - b * J[n - 1] - c * J[n - 2];
            S[n] = J[n - 2] - b * S[n - 1] - c * S[n - 2];
        }
    } else {
        // backward recurrences from n = 27 with zero start
        // (Int_analytical.f90:137-158,177-183,201-206)
        const RB ic = (RB)(1.0 / c), rb = (RB)b;
        const RB uem = (RB)(ue - ub), uep = (RB)(ue + ub);
        RB i1 = 0, i2 = 0, j1 = 0, j2 = 0, s1 = 0, s2 = 0;
#pragma unroll
        for (int m = 27; m >= 2; --m) {
            const RB base = ((m + 1) % 2 == 0) ? uem : uep;  // ue - (-1)^(m+1) ub
            const RB im = ic * RB(1.0 / (m + 1.0)) * (base - RB(m + 1.5) * rb * i1 - RB(m + 2.0) * i2);
            const RB jm = ic * (im - rb * j1 - j2);
            const RB sm = ic * (jm - rb * s1 - s2);
            if (m < NM) {
                I[m] = (double)im;
                J[m] = (double)jm;
                S[m] = (double)sm;
            }
            i2 = i1;
            i1 = im;
            j2 = j1;
            j1 = jm;
            s2 = s1;
            s1 = sm;
        }
    }
    mo.r0x = r0x;
    mo.r0y = r0y;
    mo.r0z = r0z;
    mo.px = px;
    mo.py = py;
    mo.pz = pz;
}

}  // namespace
}  // namespace rf
