// nse_round.hpp -- correctly rounded roots and quotients for the stencils' inner
// loops, each valid on the range its comment states.
//
// All follow P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", IBM J. Res. Dev. 34 (1990): from an approximation, one
// fused step gives the remainder exactly, and a second one adds the correction
// and rounds once; the root's approximation is refined by Goldschmidt's coupled
// iteration on the root and half of its reciprocal.
// tests/test_gpu_nse_round.py compares them with IEEE arithmetic.
#pragma once

#include <hip/hip_runtime.h>

namespace saras {
namespace nse {

// sqrtf(a) for a >= 2^-100 (11 issue slots where the library's root, which
// scales its argument near the ends of the range, takes 17); 0 for smaller and
// for negative a.
__device__ __forceinline__ float sqrt_rn(float a) {
    const float y = __builtin_amdgcn_rsqf(a);
    float g = a * y, h = 0.5f * y;
    const float e = fmaf(-h, g, 0.5f);
    g = fmaf(g, e, g);
    h = fmaf(h, e, h);
    return a < 0x1p-100f ? 0.0f : fmaf(fmaf(-g, g, a), h, g);
}

// a / b from the correctly rounded reciprocal y of b, for quotients and
// remainders that are no subnormal numbers (3 issue slots, the division's 11)
__device__ __forceinline__ float quot_rn(float a, float b, float y) {
    const float q = a * y;
    return fmaf(fmaf(-b, q, a), y, q);
}
// ... with the reciprocal by one step from the hardware's, for b of 2^-60 to
// 2^120 (6 issue slots)
__device__ __forceinline__ float quot_rn(float a, float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    return quot_rn(a, b, fmaf(fmaf(-b, y, 1.0f), y, y));
}

// a / 6 in four instructions (v_div_fixup gives infinities and NaN their
// quotients); a subnormal quotient may differ by one unit
__device__ __forceinline__ double by6(double a) {
    const double y = 1.0 / 6.0, q = a * y;
    return __builtin_amdgcn_div_fixup(fma(fma(-6.0, q, a), y, q), 6.0, a);
}

}  // namespace nse
}  // namespace saras
