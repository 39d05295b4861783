// kernel_eval.h -- inline kernel-entry evaluation for the HIP kernels.
//
// K(i,j) = k(||x1_i - x2_j||) on Morton-sorted indices, plus the regularization
// when the sorted indices coincide (reference: kernel_system_assembler.h:38-52,
// 82-96).  r^2 is accumulated as r2 = r2 + t*t in dimension order, exactly like
// the CPU restatement; exp/sqrt/yn come from the ROCm device library.
#pragma once
#include "hmg_internal.h"

namespace hmg {

__device__ __forceinline__ double dist2(const Coords& a, int i, const Coords& b, int j, int dim)
{
    double r2 = 0.0;
#pragma unroll
    for (int d = 0; d < MAX_POINT_DIMENSION; d++) {
        if (d < dim) {
            double t = a.x[d][i] - b.x[d][j];
            r2 = __dadd_rn(r2, __dmul_rn(t, t));
        }
    }
    return r2;
}

// One kernel kind fixed at compile time: code for one kind only, which keeps the
// register count of kernels that evaluate entries in their inner loops low (the
// Bessel function of the Matern kernel alone needs many registers).
template <int KIND>
__device__ __forceinline__ double kernel_of_r2_k(const KernelParams& kp, double r2)
{
    if (KIND == HMG_KERNEL_GAUSSIAN_REF) {
        const double r = sqrt(r2);
        return exp(-(r * r));
    }
    if (KIND == HMG_KERNEL_MATERN_REF) {
        const double r = sqrt(r2);
        return (yn(1, r + 1.0e-15) * r) / kp.c1;
    }
    if (KIND == HMG_KERNEL_GAUSSIAN) return exp(-(r2 * kp.c0));
    if (KIND == HMG_KERNEL_EXPONENTIAL) return exp(-(sqrt(r2) * kp.c0));
    return __builtin_nan("");
}

// e^x for x <= 0 (the argument of the product kernels' entries), within 1 ulp:
// Cody-Waite reduction x = n ln2 + r with ln2 split into two doubles (its double
// and the double of the remainder), |r| <= ln2/2, then a polynomial of degree 12
// by Horner's rule, scaled by 2^n.  n is read off the low word of x log2(e) + 1.5 2^52.
// The polynomial is 1 + r + r^2/2 + r^3 q(r), q the interpolant of the remainder in the
// ten Chebyshev nodes of the interval (10^-18 relative; the Taylor polynomial needs one
// degree more for 4 10^-18).  Arguments below -800 give 0 (e^-800 is below the
// smallest double).
__device__ __forceinline__ double exp_nonpos(double x)
{
    x = fmax(x, -800.0);
    const double m = __fma_rn(x, 1.4426950408889634, 6755399441055744.0);
    const double n = m - 6755399441055744.0;
    double r = __fma_rn(n, -0.6931471805599453, x);
    r = __fma_rn(n, -2.3190468138462996e-17, r);
    double p = 2.0911229798760165e-09;
    p = __fma_rn(p, r, 2.5100375929185925e-08);
    p = __fma_rn(p, r, 2.755728298391084e-07);
    p = __fma_rn(p, r, 2.7557268480106926e-06);
    p = __fma_rn(p, r, 2.480158731713526e-05);
    p = __fma_rn(p, r, 0.00019841269863040675);
    p = __fma_rn(p, r, 0.0013888888888886554);
    p = __fma_rn(p, r, 0.008333333333330065);
    p = __fma_rn(p, r, 0.041666666666666664);
    p = __fma_rn(p, r, 0.16666666666666669);
    p = __fma_rn(p, r, 0.5);
    p = __fma_rn(p, r, 1.0);
    p = __fma_rn(p, r, 1.0);
    return ldexp(p, __double2loint(m));
}

// sqrt(x) for finite x >= 0: the hardware reciprocal square root (relative error at most
// 2^-24.2 in 8.4 10^9 random arguments on MI355X; its infinity at 0 made finite), a
// Goldschmidt step and one Newton correction of the root, g += (x - g^2) h with the
// unrefined h, whose error is its final rounding but for 2^-13 ulp or so: 214 of those
// arguments were rounded to the other neighbour, none with a refined h or a second
// correction.  (An entry's error is that of the exponential: at most 0.86 ulp in all, 0.89
// with the exact root and the longer exponential.)
__device__ __forceinline__ double sqrt_nonneg(double x)
{
    const double y = fmin(__builtin_amdgcn_rsq(x), 1.0e300);
    double g = x * y;
    const double h = 0.5 * y;
    const double r = __fma_rn(-g, h, 0.5);
    g = __fma_rn(g, r, g);
    const double d = __fma_rn(-g, g, x);
    return __fma_rn(d, h, g);
}

// The entries of the FP64 products (near field, dense rows, stored near field):
// the Gaussian and exponential kernels through exp_nonpos / sqrt_nonneg (fewer
// instructions than the general functions: no overflow, scaling or class
// handling), the reference kernels as above.  The ACA keeps kernel_of_r2_k.
template <int KIND>
__device__ __forceinline__ double kernel_of_r2_prod(const KernelParams& kp, double r2)
{
    if (KIND == HMG_KERNEL_GAUSSIAN) return exp_nonpos(-(r2 * kp.c0));
    if (KIND == HMG_KERNEL_EXPONENTIAL) return exp_nonpos(-(sqrt_nonneg(r2) * kp.c0));
    return kernel_of_r2_k<KIND>(kp, r2);
}

__device__ __forceinline__ double kernel_of_r2(const KernelParams& kp, double r2)
{
    switch (kp.kind) {
    case HMG_KERNEL_GAUSSIAN_REF:
        return kernel_of_r2_k<HMG_KERNEL_GAUSSIAN_REF>(kp, r2);
    case HMG_KERNEL_MATERN_REF:
        return kernel_of_r2_k<HMG_KERNEL_MATERN_REF>(kp, r2);
    case HMG_KERNEL_GAUSSIAN:
        return kernel_of_r2_k<HMG_KERNEL_GAUSSIAN>(kp, r2);
    case HMG_KERNEL_EXPONENTIAL:
        return kernel_of_r2_k<HMG_KERNEL_EXPONENTIAL>(kp, r2);
    default:
        return __builtin_nan("");
    }
}

__device__ __forceinline__ double kernel_entry(const KernelParams& kp, const Coords& a, int i,
                                               const Coords& b, int j)
{
    double v = kernel_of_r2(kp, dist2(a, i, b, j, kp.dim));
    if (i == j) v += kp.reg;
    return v;
}

template <int KIND>
__device__ __forceinline__ double kernel_entry_k(const KernelParams& kp, const Coords& a, int i,
                                                 const Coords& b, int j)
{
    double v = kernel_of_r2_k<KIND>(kp, dist2(a, i, b, j, kp.dim));
    if (i == j) v += kp.reg;
    return v;
}

// Host side: runs the statements with `constexpr int KIND` set to the kernel kind
// (kinds are validated when a kernel object is created).
#define HMG_DISPATCH_KIND(kind, ...)                                              \
    switch (kind) {                                                               \
    case HMG_KERNEL_GAUSSIAN_REF: {                                               \
        constexpr int KIND = HMG_KERNEL_GAUSSIAN_REF;                             \
        __VA_ARGS__;                                                              \
    } break;                                                                      \
    case HMG_KERNEL_MATERN_REF: {                                                 \
        constexpr int KIND = HMG_KERNEL_MATERN_REF;                               \
        __VA_ARGS__;                                                              \
    } break;                                                                      \
    case HMG_KERNEL_GAUSSIAN: {                                                   \
        constexpr int KIND = HMG_KERNEL_GAUSSIAN;                                 \
        __VA_ARGS__;                                                              \
    } break;                                                                      \
    default: {                                                                    \
        constexpr int KIND = HMG_KERNEL_EXPONENTIAL;                              \
        __VA_ARGS__;                                                              \
    } break;                                                                      \
    }

}  // namespace hmg
