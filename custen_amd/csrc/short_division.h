// short_division.h -- division by a value whose reciprocal is at hand: the steps
// of the GPU's IEEE division (reciprocal estimate, two Newton steps, quotient,
// remainder, one correction) without its operand scaling and special-case fixup,
// which leave operands alone while |d| lies in [2^-500, 2^500] and the quotient
// in [2^-400, finite]; within that range the bits are those of n / d.
#pragma once

#include <hip/hip_runtime.h>

namespace custen {
namespace dev {

constexpr double kMinQuotient = 0x1p-400;
constexpr double kMinDivisor = 0x1p-500, kMaxDivisor = 0x1p500;

__device__ __forceinline__ double recipOf(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}
__device__ __forceinline__ double quotient(double n, double d, double y)
{
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
}

}  // namespace dev
}  // namespace custen
