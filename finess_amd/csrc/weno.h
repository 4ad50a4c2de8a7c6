// weno.h -- fifth-order WENO reconstructions on the device.
//
// JS5 : lib/WenoReconstruct.cpp:90-141 (Jiang & Shu 1996)
// Z5  : lib/WenoReconstruct.cpp:385-438 (Borges et al. 2008)
// FD5 : lib/WenoReconstruct.cpp:580-616 (linear weights 0.1, 0.6, 0.3)
//
// g[0..4] = u_{i-2..i+2}; the result is the value at x_{i+1/2}.
//
// For the common power_param == 2 the JS weights avoid pow():
//  FP64: omega_k = d_k/a_k / sum_j d_j/a_j with a_k = (eps+beta_k)^2 is formed
//        with one division as d_k prod_{j!=k} a_j / sum_j d_j prod_{i!=j} a_i
//        (products of two a's stay inside the FP64 range for eps >= 1e-75
//        and differences of the g up to 1e37);
//  FP32: the same weights as d_k r_k / sum_j d_j r_j with r_k = min(a)/a_k in
//        [0,1], so nothing overflows and a weight that underflows is one whose
//        exact value is below FP32 resolution anyway (eps = 1e-29 gives
//        a = 1e-58, outside the FP32 range).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "fastmath.h"

namespace finess {

enum WenoKind : int {
    WENO_JS5_P2 = 0, WENO_JS5_POW = 1, WENO_Z5 = 2, WENO_FD5 = 3,
    // Z5 with power_param == 2, whose ratios are squared instead of raised
    WENO_Z5_P2 = 4,
    // the face-list path of stage2d_wide.hip
    WENO_JS7 = 5, WENO_JS9 = 6, WENO_JS11 = 7, WENO_Z7 = 8, WENO_Z9 = 9, WENO_FD7 = 10, WENO_FD9 = 11,
    WENO_O1 = 12
};

// The kind of fifth-order Z: power_param == 2 (the default) has a form without
// pow (weno5_fp64).  Its product of three denominators, the largest of them of
// the order of one, is at least about eps^2, which eps >= 1e-90 keeps in range.
__host__ __device__ constexpr int weno_z5_kind(double power, double eps)
{
    return power == 2.0 && eps >= 1e-90 ? WENO_Z5_P2 : WENO_Z5;
}

template <typename R>
struct WenoParams {
    R eps;
    R power;
};

template <typename R>
__host__ __device__ __forceinline__ void weno5_candidates(const R g[5], R& u1, R& u2, R& u3)
{
    u1 = (R(1) / R(3)) * g[0] - (R(7) / R(6)) * g[1] + (R(11) / R(6)) * g[2];
    u2 = (R(-1) / R(6)) * g[1] + (R(5) / R(6)) * g[2] + (R(1) / R(3)) * g[3];
    u3 = (R(1) / R(3)) * g[2] + (R(5) / R(6)) * g[3] - (R(1) / R(6)) * g[4];
}

template <typename R>
__host__ __device__ __forceinline__ void weno5_betas(const R g[5], R& b0, R& b1, R& b2)
{
    const R d0 = g[0] - R(2) * g[1] + g[2], e0 = g[0] - R(4) * g[1] + R(3) * g[2];
    const R d1 = g[1] - R(2) * g[2] + g[3], e1 = g[1] - g[3];
    const R d2 = g[2] - R(2) * g[3] + g[4], e2 = R(3) * g[2] - R(4) * g[3] + g[4];
    b0 = (R(13) / R(12)) * (d0 * d0) + R(0.25) * (e0 * e0);
    b1 = (R(13) / R(12)) * (d1 * d1) + R(0.25) * (e1 * e1);
    b2 = (R(13) / R(12)) * (d2 * d2) + R(0.25) * (e2 * e2);
}

template <typename R>
__host__ __device__ __forceinline__ R fmin3(R a, R b, R c)
{
    return fmin(fmin(a, b), c);
}


// Unnormalised JS5 weights for power_param == 2 (see the header comment).
__host__ __device__ __forceinline__ void js5_p2_terms(double b0, double b1, double b2, double eps,
                                                      double& t0, double& t1, double& t2)
{
    double a0 = eps + b0, a1 = eps + b1, a2 = eps + b2;
    a0 *= a0; a1 *= a1; a2 *= a2;
    t0 = 0.1 * (a1 * a2); t1 = 0.6 * (a0 * a2); t2 = 0.3 * (a0 * a1);
}
__host__ __device__ __forceinline__ void js5_p2_terms(float b0, float b1, float b2, float eps,
                                                      float& t0, float& t1, float& t2)
{
    float a0 = eps + b0, a1 = eps + b1, a2 = eps + b2;
    a0 *= a0; a1 *= a1; a2 *= a2;
    const float amin = fmin3(a0, a1, a2);
    t0 = 0.1f * (amin * frcp(a0)); t1 = 0.6f * (amin * frcp(a1)); t2 = 0.3f * (amin * frcp(a2));
}

// Nonlinear JS weights (normalised, summing to one).
template <int KIND, typename R>
__host__ __device__ __forceinline__ void weno5_weights(const R g[5], const WenoParams<R>& wp, R w[3])
{
    R b0, b1, b2;
    weno5_betas(g, b0, b1, b2);
    if (KIND == WENO_FD5) {
        w[0] = R(0.1); w[1] = R(0.6); w[2] = R(0.3);
    } else if (KIND == WENO_JS5_P2) {
        R t0, t1, t2;
        js5_p2_terms(b0, b1, b2, wp.eps, t0, t1, t2);
        const R inv = R(1) / (t0 + t1 + t2);
        w[0] = t0 * inv; w[1] = t1 * inv; w[2] = t2 * inv;
    } else if (KIND == WENO_JS5_POW) {
        const R t0 = R(0.1) * pow(wp.eps + b0, -wp.power);
        const R t1 = R(0.6) * pow(wp.eps + b1, -wp.power);
        const R t2 = R(0.3) * pow(wp.eps + b2, -wp.power);
        const R inv = R(1) / (t0 + t1 + t2);
        w[0] = t0 * inv; w[1] = t1 * inv; w[2] = t2 * inv;
    } else { // Z5
        const R tau5 = fabs(b0 - b2);
        const R t0 = R(0.1) * (R(1) + pow(tau5 / (wp.eps + b0), wp.power));
        const R t1 = R(0.6) * (R(1) + pow(tau5 / (wp.eps + b1), wp.power));
        const R t2 = R(0.3) * (R(1) + pow(tau5 / (wp.eps + b2), wp.power));
        const R inv = R(1) / (t0 + t1 + t2);
        w[0] = t0 * inv; w[1] = t1 * inv; w[2] = t2 * inv;
    }
}

// The reconstruction as the scheme's sources write it, in the arithmetic of R.
// The FP32 form, the routed FP64 form and the limited Lax-Wendroff step take
// it (the limiter decides by the signs of differences that rounding makes, so
// its step keeps the operation order it was pinned with).
template <int KIND, typename R>
__host__ __device__ __forceinline__ R weno5(const R g[5], const WenoParams<R>& wp)
{
    R u1, u2, u3;
    weno5_candidates(g, u1, u2, u3);
    if (KIND == WENO_FD5) return R(0.1) * u1 + R(0.6) * u2 + R(0.3) * u3;
    R b0, b1, b2;
    weno5_betas(g, b0, b1, b2);
    if (KIND == WENO_JS5_P2) {
        R t0, t1, t2;
        js5_p2_terms(b0, b1, b2, wp.eps, t0, t1, t2);
        return (t0 * u1 + t1 * u2 + t2 * u3) * rcp_nr(t0 + t1 + t2);
    } else if (KIND == WENO_JS5_POW) {
        const R t0 = R(0.1) * pow(wp.eps + b0, -wp.power);
        const R t1 = R(0.6) * pow(wp.eps + b1, -wp.power);
        const R t2 = R(0.3) * pow(wp.eps + b2, -wp.power);
        return (t0 * u1 + t1 * u2 + t2 * u3) / (t0 + t1 + t2);
    } else {
        const R tau5 = fabs(b0 - b2);
        const R t0 = R(0.1) * (R(1) + pow(tau5 / (wp.eps + b0), wp.power));
        const R t1 = R(0.6) * (R(1) + pow(tau5 / (wp.eps + b1), wp.power));
        const R t2 = R(0.3) * (R(1) + pow(tau5 / (wp.eps + b2), wp.power));
        return (t0 * u1 + t1 * u2 + t2 * u3) / (t0 + t1 + t2);
    }
}

// The FP64 reconstruction, on the differences d_i = g[i+1] - g[i].
//
// The indicators are quadratic forms of two neighbouring differences,
//     beta_0 = 4/3 (d0^2 - 11/4 d0 d1 + 5/2 d1^2),
//     beta_1 = 4/3 (d1^2 -  5/4 d1 d2 +     d2^2),
//     beta_2 = 4/3 (d3^2 - 11/4 d3 d2 + 5/2 d2^2),
// (the outer forms' eigenvalues are 0.18 and 3.3, so their cancellation costs at
// most a factor of 18), and the candidates are g[2] plus two of them.
// The common factor 4/3 leaves every weight ratio unchanged, so it is dropped
// and eps is scaled by 3/4 instead.  The reconstruction of a fused stage takes
// 36 FP64 instructions and one reciprocal estimate, where the form above takes
// 55 (candidates of five values, indicators as sums of squares).
//
// power_param == 2: JS multiplies by the other two a_k (see the header); Z
// (WENO_Z5_P2) forms its three ratios tau / (eps + beta_k) from the
// reciprocal of the product of the denominators, scaled to the order of one
// (without the scaling the product overflows from differences of 1e51 on; it
// costs 3 to 4% of a stage: Euler 1024^2 65.2 -> 67.9 us, 390 with pow).
template <int KIND>
__host__ __device__ __forceinline__ double weno5_fp64(const double g[5], double eps, double power)
{
    // every multiply-add is written out: g[i] that are products of the caller
    // are not drawn into the differences in one kernel and left alone in another
#pragma clang fp contract(off)
    const double d0 = g[1] - g[0], d1 = g[2] - g[1], d2 = g[3] - g[2], d3 = g[4] - g[3];
    if (KIND == WENO_FD5)
        return g[2] + fma(11.0 / 60.0, d1, fma(24.0 / 60.0, d2, fma(-2.0 / 60.0, d0, (-3.0 / 60.0) * d3)));
    const double e = 0.75 * eps;
    const double c1 = scalar_const(-2.75), c2 = scalar_const(-1.25), c3 = scalar_const(2.5);
    const double p1 = d1 * d1, p2 = d2 * d2;
    const double a0 = fma(d0, fma(c1, d1, d0), fma(c3, p1, e));
    const double a1 = fma(d1, fma(c2, d2, d1), fma(d2, d2, e));
    const double a2 = fma(d3, fma(c1, d2, d3), fma(c3, p2, e));
    // candidate minus g[2], times its linear weight over 0.1 (1, 6 and 3)
    const double v0 = fma(5.0 / 6.0, d1, (-1.0 / 3.0) * d0);
    const double v1 = fma(2.0, d2, d1);
    const double v2 = fma(2.0, d2, -0.5 * d3);
    double t0, t1, t2;  // unnormalised weights without their 0.1, 0.6, 0.3
    if (KIND == WENO_JS5_P2) {
        const double s0 = a0 * a0, s1 = a1 * a1, s2 = a2 * a2;
        t0 = s1 * s2; t1 = s0 * s2; t2 = s0 * s1;
    } else if (KIND == WENO_JS5_POW) {
        t0 = pow(a0, -power); t1 = pow(a1, -power); t2 = pow(a2, -power);
    } else if (KIND == WENO_Z5_P2) {
        // the ratios do not change with a common factor: a power of two brings the
        // denominators to the order of one, so that no product of them overflows
        const int n = -exponent(a0 + a2);
        const double b0 = ldexp(a0, n), b1 = ldexp(a1, n), b2 = ldexp(a2, n);
        const double q01 = b0 * b1, q12 = b1 * b2, q02 = b0 * b2;
        const double r = fabs(b0 - b2) * rcp_d(q01 * b2);
        const double z0 = r * q12, z1 = r * q02, z2 = r * q01;
        t0 = fma(z0, z0, 1.0); t1 = fma(z1, z1, 1.0); t2 = fma(z2, z2, 1.0);
    } else {
        const double tau = fabs(a0 - a2);
        t0 = 1.0 + pow(tau / a0, power); t1 = 1.0 + pow(tau / a1, power); t2 = 1.0 + pow(tau / a2, power);
    }
    const double den = fma(6.0, t1, fma(3.0, t2, t0));
    const double num = fma(t1, v1, fma(t2, v2, t0 * v0));
    return fma(num, rcp_d(den), g[2]);
}

} // namespace finess
