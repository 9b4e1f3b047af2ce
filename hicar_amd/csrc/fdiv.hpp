// Correctly rounded FP32 division in three operations once a reciprocal is
// known, for operands in a range where no step over- or underflows.
//
// With y the reciprocal of d and q0 = RN(x*y), the remainder x - q0*d is
// exactly representable and one FMA gives it; q = RN(q0 + (x - q0*d)*y) is
// then the correctly rounded quotient RN(x/d) when y is within half an ulp
// of 1/d and q0 within one ulp of x/d (Markstein, "IA-64 and Elementary
// Functions", 2000, theorem 8.10; Cornea, Harrison and Tang, "Scientific
// Computing on Itanium-based Systems", 2002, ch. 8).  The reciprocal here is
// the hardware estimate (v_rcp_f32, 1 ulp) refined by one Newton step.  The
// library does not rely on the theorem's premises holding for that y:
// icar_adv_verify_division compares the quotient with the IEEE division for
// every pair of significands on the device, and the kernels take this path
// only inside the range where every operation scales exactly with the
// operands' exponents, so the significand pairs cover all of
// it.
//
// The remainder is formed negated, rn = q0*d - x, and the quotient as
// q0 - rn*y: for d > 0 a zero numerator then keeps its sign (+0 / d = +0,
// -0 / d = -0), as the IEEE division does.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace icaradv {

// 1/d: the hardware estimate and one Newton step, e = 1 - d*y0, y = y0 + e*y0
__device__ __forceinline__ float recip_nr(float d)
{
    const float y0 = __builtin_amdgcn_rcpf(d);
    const float e = __builtin_fmaf(-d, y0, 1.0f);
    return __builtin_fmaf(e, y0, y0);
}

// RN(x/d) from y = recip_nr(d), for operands in range (below)
__device__ __forceinline__ float div_y(float x, float d, float y)
{
    const float q0 = x * y;
    const float rn = __builtin_fmaf(q0, d, -x);
    return __builtin_fmaf(-rn, y, q0);
}

// The quotient is taken where the divisor is positive and in [2^-60, 2^60] and
// the numerator zero or at least 2^-101 (a kernel's own bounds lie inside
// these), so that 1/d, x*y and the quotient are normal numbers and the
// remainder is exact: every step then equals, scaled by a power of two, the
// same step on the operands' significands.  The device check covers the
// reciprocal's scaling over d's exponents FDIV_E_LO..FDIV_E_HI.
constexpr int FDIV_E_LO = -60, FDIV_E_HI = 60;

// The key of a numerator by which the kernels find the smallest non-zero one
// of a group: 2*bits - 1 unsigned, so that +-0 maps to the largest value and
// never counts as small
__device__ __forceinline__ uint32_t nz_key(float x)
{
    return (__float_as_uint(x) << 1) - 1u;
}

}  // namespace icaradv
