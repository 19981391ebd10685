// FP64 quotients that share a denominator, on the device.
#pragma once
#include <hip/hip_runtime.h>

namespace pppm_amd
{

// 1 / d for quotients that share the denominator d: the reciprocal estimate and two Newton steps,
// then per quotient the product, its residual and the correction. These are the steps of the
// compiler's own FP64 division without its range scaling, so the quotients are its bits (the
// correctly rounded ones) as long as neither operand nor quotient comes near the exponent limits;
// the caller sees to that.
// The fixup gives zeros, infinities and NaN among n and d their IEEE results.
__device__ inline double shared_rcp(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
}
// the same, in scalar registers, for a d that is the same in all lanes
__device__ inline double uniform_rcp(double d)
{
    const double y = shared_rcp(d);
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(y)),
                            __builtin_amdgcn_readfirstlane(__double2loint(y)));
}
__device__ inline double shared_div(double n, double d, double y)
{
    const double m = n * y;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d, m, n), y, m), d, n);
}

}  // namespace pppm_amd
