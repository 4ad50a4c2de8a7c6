// fastmath.h -- reciprocal, division and square root of the device code.
// The FP32 form keeps its values to FP32 resolution, so the IEEE division and
// square-root sequences (about ten instructions each) are replaced by the
// hardware estimates (within one ulp).  The FP64 overloads of div_lp and
// sqrt_lp keep the IEEE operations; the fused FP64 kernels take rcp_d,
// rsqrt_d and sqrt_d, the hardware estimate and one third-order step.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace finess {

__host__ __device__ __forceinline__ float frcp(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}

// 1/x to full FP64 accuracy (within an ulp) without the IEEE division
// sequence: hardware reciprocal estimate refined by two Newton steps.
__host__ __device__ __forceinline__ double rcp_nr(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
#else
    return 1.0 / x;
#endif
}
__host__ __device__ __forceinline__ float rcp_nr(float x) { return frcp(x); }

// 1/x in FP64: the hardware estimate (about 24 bits) and one third-order
// step, r (1 + e + e^2) with e = 1 - x r, whose error e^3 lies below the last
// bit: three fused multiply-adds where two Newton steps take four.
__host__ __device__ __forceinline__ double rcp_d(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
#else
    return 1.0 / x;
#endif
}

// 1/sqrt(x) in FP64: the hardware estimate and one third-order step,
// y (1 + h/2 + 3 h^2/8) with h = 1 - x y^2.  Negative x: NaN.
__host__ __device__ __forceinline__ double rsqrt_d(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rsq(x);
    const double h = fma(-(x * y), y, 1.0);
    return fma(y * h, fma(0.375, h, 0.5), y);
#else
    return 1.0 / sqrt(x);
#endif
}

// sqrt(x), x >= 0, through rsqrt_d.  The 1e-300 keeps the reciprocal root of a
// zero finite (sqrt(0) is 1e-150) and is lost in any other value.
__host__ __device__ __forceinline__ double sqrt_d(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = x + 1e-300;
    return y * rsqrt_d(y);
#else
    return sqrt(x);
#endif
}

// The binary exponent of x as frexp takes it (x 2^-exponent in [1/2, 1)).
__host__ __device__ __forceinline__ int exponent(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_frexp_exp(x);
#else
    int e;
    (void)frexp(x, &e);
    return e;
#endif
}

// An FP64 constant held in scalar registers.  Left as a literal it ties the
// multiply-add to the two-operand form, which overwrites its addend: the
// compiler then copies every addend that is used again (five copies for each
// reconstruction, 8% of the instructions of a fused FP64 face).
__host__ __device__ __forceinline__ double scalar_const(double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+s"(c));
#endif
    return c;
}

// a / b: IEEE in FP64, a times the reciprocal estimate in FP32.
__host__ __device__ __forceinline__ double div_lp(double a, double b) { return a / b; }
__host__ __device__ __forceinline__ float div_lp(float a, float b) { return a * frcp(b); }

// sqrt: IEEE in FP64, the hardware square root (within one ulp) in FP32.
__host__ __device__ __forceinline__ double sqrt_lp(double x) { return sqrt(x); }
__host__ __device__ __forceinline__ float sqrt_lp(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_sqrtf(x);
#else
    return sqrtf(x);
#endif
}

} // namespace finess
