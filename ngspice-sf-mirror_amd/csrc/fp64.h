/*
 * Double-precision helpers of the factorization kernels.
 */
#ifndef NGMI_FP64_H
#define NGMI_FP64_H

#include <hip/hip_runtime.h>

namespace ngmi {

/* 1 / p for finite p != 0 (NaN for zero and the infinities, where 1 / p is
 * infinite or zero): v_rcp_f64 of the mantissa (2^-24) with two Newton steps,
 * the second on the exact remainder; the rounded reciprocal wherever that is a
 * normal number, without the scaled division sequence's branch for the range's
 * ends */
__device__ __forceinline__ double recip(double p)
{
    const double m = __builtin_amdgcn_frexp_mant(p);
    double r = __builtin_amdgcn_rcp(m);
    r = fma(fma(-m, r, 1.0), r, r);
    r = fma(fma(-m, r, 1.0), r, r);
    return __builtin_amdgcn_ldexp(r, -__builtin_amdgcn_frexp_exp(p));
}

/* a / b from r = 1 / b as rounded: one correction of a r by its exact
 * remainder gives the rounded quotient (Markstein 1990) while no step under-
 * or overflows; off the dependent chain of a full division */
__device__ __forceinline__ double div_by(double a, double b, double r)
{
    const double q = a * r;
    return fma(fma(-q, b, a), r, q);
}

/* where div_by's steps stay normal.  Elsewhere (overflow to infinity,
 * subnormal pivots, negative zeros, whose sign the correction loses) the
 * quotient is a true division's. */
__device__ __forceinline__ bool div_by_divisor(double b) { return fabs(b) > 0x1p-400 && fabs(b) < 0x1p400; }
__device__ __forceinline__ bool div_by_dividend(double a) { return fabs(a) > 0x1p-500 && fabs(a) < 0x1p500; }

}  // namespace ngmi

#endif
