// Single-operation IEEE-754 binary32 arithmetic for device code.
//
// The quantiser must reproduce CPU arithmetic bit for bit, so every f32 step has to be exactly one
// correctly rounded operation.  Plain C operators give that under two conditions this build enforces:
// contraction is off (-ffp-contract=off on the command line and the pragma below, so a*b+c is never
// fused) and division / square root are the correctly rounded forms
// (-fhip-fp32-correctly-rounded-divide-sqrt, the compiler's default, named explicitly in the Makefile).
// HIP's __fsqrt_rn is NOT used: without OCML_BASIC_ROUNDED_OPERATIONS it maps to the approximate
// hardware square root.
#pragma once
#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace bitnet {
__device__ __forceinline__ float f32_add(float a, float b) { return a + b; }
__device__ __forceinline__ float f32_mul(float a, float b) { return a * b; }
__device__ __forceinline__ float f32_div(float a, float b) { return a / b; }
__device__ __forceinline__ float f32_sqrt(float a) { return __builtin_sqrtf(a); }

// x / d for a positive divisor d shared by many dividends.  recip must be the correctly rounded 1/d (one IEEE
// division).  q0 = RN(x*recip) is within one ulp of x/d; the remainder x - d*q0 is then exact in one FMA and
// the corrected quotient RN(q0 + rem*recip) is the correctly rounded x/d (Markstein's division step).  The
// theorem excludes divisors whose significand is all ones and needs the intermediate values to stay normal:
// invariant_divisor_ok(d) is tested once per divisor, dividend_ok(x) per dividend (zero is fine, tiny, huge
// and non-finite values are not); where either fails the caller uses the plain division.  Three operations
// per element instead of the full IEEE sequence, same bits.
__device__ __forceinline__ bool invariant_divisor_ok(float d)
{
    const unsigned bits = __builtin_bit_cast(unsigned, d);
    const unsigned expo = (bits >> 23) & 0xffu;
    return (bits >> 31) == 0u && (bits & 0x7fffffu) != 0x7fffffu && expo > 64u && expo < 190u;
}
__device__ __forceinline__ bool dividend_ok(float x)
{
    const unsigned mag = __builtin_bit_cast(unsigned, x) & 0x7fffffffu;
    return mag == 0u || (mag >= (64u << 23) && mag < (190u << 23));  // 0, or 2^-63 <= |x| < 2^63
}
// SIGNED_ZERO false: a zero dividend may lose its sign (one operation less, for callers that round to an integer next).
template <bool SIGNED_ZERO = true>
__device__ __forceinline__ float div_by_invariant_unchecked(float x, float d, float recip)
{
    const float q0 = x * recip;
    const float rem = __builtin_fmaf(-q0, d, x);
    const float q = __builtin_fmaf(rem, recip, q0);
    return SIGNED_ZERO ? __builtin_copysignf(q, x) : q;  // d > 0: the quotient has x's sign (also for -0)
}

// The correctly rounded 1/d of a divisor that invariant_divisor_ok accepts: the hardware's approximation (within one ulp)
// and one Newton step (Markstein: correctly rounded from there except for a significand of all ones).  Three dependent
// operations in place of the nine of the full division.  Compared with 1.0f / d for every float of the accepted
// exponents on the device: no difference.
__device__ __forceinline__ float recip_of_ok_divisor(float d)
{
    const float r = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}

// The one significand that invariant_divisor_ok excludes.
__device__ __forceinline__ bool significand_ok(float d) { return (__builtin_bit_cast(unsigned, d) & 0x7fffffu) != 0x7fffffu; }

// A divisor shared by many dividends, ready for use.
struct Divisor {
    float d, recip;
    bool fast;
};
__device__ __forceinline__ Divisor make_divisor(float d)
{
    Divisor v;
    v.d = d;
    v.fast = invariant_divisor_ok(d);
    v.recip = recip_of_ok_divisor(d);  // not used unless fast
    return v;
}
// x / d for values that are the same in every lane of the wavefront (or where a full division in all lanes is as cheap).
__device__ __forceinline__ float div_uniform(float x, const Divisor &v)
{
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(v.fast && dividend_ok(x))) == 0, 1)) return div_by_invariant_unchecked(x, v.d, v.recip);
    return f32_div(x, v.d);
}

// Square root for exponents 2^-62 .. 2^62: Goldschmidt's iteration from the hardware's reciprocal square root with a final
// residual correction (Markstein).  Compared with the correctly rounded root for every float of that range on the device:
// no difference.
__device__ __forceinline__ float sqrt_in_range(float a)
{
    const float r = __builtin_amdgcn_rsqf(a);
    float g = a * r, h = 0.5f * r;
    const float e = __builtin_fmaf(-h, g, 0.5f);
    g = __builtin_fmaf(g, e, g);
    h = __builtin_fmaf(h, e, h);
    return __builtin_fmaf(__builtin_fmaf(-g, g, a), h, g);
}
// The square root of a value that is the same in every lane: the plain one outside that range.
__device__ __forceinline__ float sqrt_uniform(float a)
{
    const unsigned expo = __builtin_bit_cast(unsigned, a) >> 23;  // the sign counts as a large exponent
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(expo > 64u && expo < 190u)) == 0, 1)) return sqrt_in_range(a);
    return f32_sqrt(a);
}
}  // namespace bitnet
