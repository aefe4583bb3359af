// Exact FP64 division with a reciprocal reused across numerators, shared by
// the factorisation and solve kernels.
#pragma once
#include "nrocm_internal.hpp"

namespace nrocm_div {

// hipcc expands an f64 x / d as s = div_scale(d), y = rcp(s) refined by two
// Newton steps, q0 = x' * y, r = fma(-s, q0, x'), q = div_fmas(r, y, q0),
// div_fixup(q, d, x).  When 2^-100 <= |d| <= 2^100 and 2^-900 <= |x| <= 2^600
// both scalings are identities, div_fmas is a plain fma and the fixup returns
// q unchanged, so div_with(x, d, recip_refined(d)) is bit-identical to x / d.
// Outside that range (zeros, infinities, NaNs, extreme exponents) callers use
// x / d.
__device__ __forceinline__ double recip_refined(double d)
{
    const double r0 = __builtin_amdgcn_rcp(d);
    const double e0 = __builtin_fma(-d, r0, 1.0);
    const double r1 = __builtin_fma(r0, e0, r0);
    const double e1 = __builtin_fma(-d, r1, 1.0);
    return __builtin_fma(r1, e1, r1);
}

__device__ __forceinline__ double div_with(double x, double d, double y)
{
    const double q0 = x * y;
    const double rem = __builtin_fma(-d, q0, x);
    return __builtin_fma(rem, y, q0);
}

__device__ __forceinline__ bool div_den_ok(double d)
{
    const double ad = __builtin_fabs(d);
    return ad >= 0x1p-100 && ad <= 0x1p100;
}

__device__ __forceinline__ bool div_num_ok(double x)
{
    const double ax = __builtin_fabs(x);
    return ax >= 0x1p-900 && ax <= 0x1p600;
}

// Numerator range of div_with from the exponent field alone: 2^-900 <= |x| <
// 2^600, or +0 (there q0 = +0 * y already carries x / d's sign, and rem = +0
// times y adds a zero of that sign).
__device__ __forceinline__ bool num_in_range(double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned e = (unsigned)(b >> 52) & 0x7ffu;
    return (e - 123u) <= 1499u || b == 0ull;
}

}  // namespace nrocm_div
