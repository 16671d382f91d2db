/*
 * Double-precision helpers of the factorization kernels.
 */
#ifndef NGMI_FP64_H
#define NGMI_FP64_H

#include <hip/hip_runtime.h>

namespace ngmi {

/* 1 / p: v_rcp_f64 of the mantissa (2^-24) with two Newton steps, the second
 * on the exact remainder: equal to 1.0 / p for every one of 2.6e8 random
 * mantissas, without the scaled division sequence's branch for the range's
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
 * remainder gives the rounded quotient (Markstein 1990) while neither
 * under- nor overflows; off the dependent chain of a full division */
__device__ __forceinline__ double div_by(double a, double b, double r)
{
    const double q = a * r;
    return fma(fma(-q, b, a), r, q);
}

}  // namespace ngmi

#endif
