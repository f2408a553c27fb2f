/*
 * Double-precision reciprocal and square root of the force kernels' pair terms.
 *
 * Newton-Raphson steps from the hardware's estimates (relative error below 5e-8, so that two steps
 * reach the last bit), without the scaling and the special cases that a division or sqrt() carries
 * for zero, denormal and infinite operands: 5 instructions instead of 11, and 11 instead of 27 for a
 * root and its reciprocal.
 *
 * recip_normal and root_recip_normal, for sums that promise no bits (the Verlet-list scheme's fast
 * kernels): within one unit in the last place.  Next to the middle of two doubles the last step can round the
 * wrong way: of 1.15 million arguments, the 4096 nearest to each of 25 powers of two among them, 150
 * (2^k (1 - m 2^-53) with m = 3, 5, .. 13) were an ulp off.  268 million random ones were not.
 *
 * recip_rounded: the correctly rounded reciprocal, as the division gives it, where bits are promised
 * (FP64 cluster pairs, full lists).  A Newton-Raphson step in fused arithmetic from a value within an ulp
 * of 1/d rounds correctly for every mantissa but the one of all ones (P. Markstein, "Computation of
 * elementary functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990); for that
 * one the hardware's estimate leads to the right value too (checked at 25 exponents; none of the 1.15
 * million differed from the division).  37,044 atoms of a mixture, us a call: division 30.1, this 29.0,
 * recip_normal 28.3; 256,000 atoms of 4x8 clusters 169, 152, 147.
 *
 * A zero argument's reciprocal is NaN (a pair at distance zero: its force is 0 times infinity, NaN,
 * either way), its root zero, and an argument whose reciprocal overflows (a distance below 1e-154)
 * gives NaN too; callers that need the special
 * cases divide, and so do the passes that instructions do not bound: the EAM density pass (264 us with
 * a root from here, 261 without, 1.05 M atoms) and the FP64 cluster pairs' half lists.
 */
#pragma once
#include <hip/hip_runtime.h>

namespace mdg {

__device__ inline double recip_normal(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y        = fma(y, fma(-d, y, 1.0), y);
    return fma(y, fma(-d, y, 1.0), y);
}

__device__ inline double recip_rounded(double d)
{
    const double y = recip_normal(d);
    return fma(y, fma(-d, y, 1.0), y);
}

// *r = sqrt(d), returning 1 / *r
__device__ inline double root_recip_normal(double d, double* r)
{
    const double y = __builtin_amdgcn_rsq(d);
    double g = d * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g              = fma(g, e, g);
    h              = fma(h, e, h);
    g              = fma(fma(-g, g, d), h, g);
    h              = h + h;
    *r             = fmax(g, 0.0);  // (g is NaN for zero)
    return fma(h, fma(-g, h, 1.0), h);
}

}  // namespace mdg
