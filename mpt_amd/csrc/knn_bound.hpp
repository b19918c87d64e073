// The exact metric distance and the FP32 bounds in front of it, shared by the
// nearest-neighbour kernels.
//
// Prefilter soundness.  With u = 2^-24, S = max|q| + max|p| and
// eps = 2.01 u S, each FP32 coordinate difference satisfies
// |t_i - (q_i - p_i)| <= eps.  For L2 (squared distances d):
//   |d32 - d| <= 2 eps sqrt(D d) + D eps^2 + g_D (d + 2 eps sqrt(D d) + D eps^2),
//   g_D = D u / (1 - D u)
// and for L1: |d32 - d| <= D eps + g_D (d + D eps).  A node can enter the
// list only if d <= T (T = current k-th distance, squared for L2), hence only
// if d32 <= T + eta(T).  The kernels use 2 * eta plus a relative 2^-40 for
// the sqrt rounding of list entries.
#pragma once
#include "internal.hpp"

namespace mptg {
namespace {

// FP64 metric value, left-to-right, no contraction (matches the oracle).
template <int D, int METRIC>
__device__ __forceinline__ double exact_dist(const double* __restrict__ a, const double* __restrict__ b) {
    double s = 0.0;
    if constexpr (METRIC == MPTG_METRIC_L1) {
#pragma unroll
        for (int i = 0; i < D; ++i) s = s + __builtin_fabs(a[i] - b[i]);
        return s;
    } else {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            double t = a[i] - b[i];
            s = s + t * t;
        }
        return __builtin_sqrt(s);
    }
}

// Prefilter threshold in the prefilter's units (squared distance for L2,
// distance for L1) from the list's k-th distance `dk` (metric value).
template <int D, int METRIC>
__device__ __forceinline__ float prefilter_threshold(double dk, double S) {
    if (!__builtin_isfinite(dk)) return __builtin_inff();
    const double u = 0x1.0p-24;
    const double eps = 2.01 * u * S;
    const double g = D * u / (1.0 - D * u);
    double T, eta;
    if constexpr (METRIC == MPTG_METRIC_L1) {
        T = dk;
        eta = D * eps + g * (T + D * eps);
    } else {
        T = dk * dk;
        double r = 2.0 * eps * __builtin_sqrt(D * T) + D * eps * eps;
        eta = r + g * (T + r);
    }
    double thr = T * (1.0 + 0x1.0p-40) + 2.0 * eta + 1e-300;
    float f = (float)thr;
    // round up (thr > 0) so that the FP32 comparison never undercuts the FP64 bound
    return (double)f < thr ? float_of(bits_of(f) + 1u) : f;
}

// An upper bound, in metric units, on the exact distance of a node whose
// prefilter value (FP32 sum, squared for L2) is `a`: the inverse of the
// error bound behind prefilter_threshold.  L1: |a - d| <= D eps + g (d +
// D eps) gives d <= (a + D eps (1 + g)) / (1 - g).  L2: |a - T| <= r + g (T +
// r) with r = 2 eps sqrt(D T) + D eps^2 gives, for x = sqrt(T), (1 - g) x^2
// - 2 (1 + g) eps sqrt(D) x - (a + (1 + g) D eps^2) <= 0, bounded by the
// quadratic's larger root.  A relative 2^-40 covers the FP64 rounding.
template <int D, int METRIC>
__device__ __forceinline__ double prefilter_upper(float a, double S) {
    const double u = 0x1.0p-24;
    const double eps = 2.01 * u * S;
    const double g = D * u / (1.0 - D * u);
    double x;
    if constexpr (METRIC == MPTG_METRIC_L1) {
        x = ((double)a + D * eps * (1.0 + g)) / (1.0 - g);
    } else {
        const double bq = (1.0 + g) * eps * __builtin_sqrt((double)D);
        const double c = (double)a + (1.0 + g) * D * eps * eps;
        x = (bq + __builtin_sqrt(bq * bq + (1.0 - g) * c)) / (1.0 - g);
    }
    return x * (1.0 + 0x1.0p-40) + 1e-300;
}

}  // namespace
}  // namespace mptg
