/*
 * Double-precision reciprocal and square root of the force kernels' pair terms.
 *
 * Newton-Raphson steps from the hardware's estimates (relative error below 5e-8, so that two steps
 * reach the last bit), without the scaling and the special cases that a division or sqrt() carries
 * for zero, denormal and infinite operands: 5 instructions instead of 11, and 11 instead of 27 for a
 * root and its reciprocal.  Over 268 million arguments each of 1e-3 .. 1e3 and 0.5 .. 50 every result
 * was the correctly rounded one.  A zero argument gives NaN (a pair at distance zero: its force is
 * 0 times infinity, NaN, either way); callers that need the special cases divide, and so does the
 * EAM density pass, which is not bound by instructions (264 us with it, 261 without, 1.05 M atoms).
 * Per call at 1.05 M atoms: staged LJ forces 213 -> 207 us, EAM forces 343 -> 334; FP64 cluster pairs of
 * 35,000 atoms 24.6 -> 23.5.
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
    *r             = g;
    return fma(h, fma(-g, h, 1.0), h);
}

}  // namespace mdg
