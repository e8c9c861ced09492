// fp64.hpp — short correctly rounded fp64 division and square root for operands
// in known, moderate ranges (the Jacobi rotation's scalar chain).
//
// For a / b and sqrt(x) the compiler emits a refinement of the hardware
// reciprocal (v_rcp_f64) or reciprocal square root (v_rsq_f64) wrapped in range
// handling: v_div_scale / v_div_fmas / v_div_fixup for division, and a 2^256
// pre-scale of tiny inputs plus a class check for 0 and inf for sqrt. The helpers
// below keep the refinement and drop the wrapping, so on operands that never need
// it they return the same bits as IEEE `/` and `sqrt` in fewer dependent steps:
//   * div_rn(a, b): two Newton-Raphson steps r <- r + r (1 - b r) on the
//     reciprocal, then q = a r corrected once by the exact residual a - b q
//     (Markstein's correctly rounded quotient). Needs b and a / b normal and far
//     from overflow, which holds for |b| in [2^-900, 2^900] and |a| < 2^900.
//   * sqrt_and_rcp(x, g, r): both sqrt(x) and 1 / sqrt(x), from one iteration.
// slime_probe_fp64_core (probe.hip) checks them against `/` and `sqrt` bit for bit on the
// device, over exponents from 2^-40 up (x) and in [-60, 60] (a, b), and the whole
// rotation against its IEEE form; that form's own error is checked on the host
// (tests/jacobi_wave_check.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include "jacobi_wave.hpp"

namespace slime {

__device__ __forceinline__ double div_rn(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// g = sqrt(x) and r = 1 / sqrt(x) with both IEEE roundings (the bits of `sqrt(x)` and
// `1.0 / sqrt(x)`), for x in [2^-40, 2^900), where no pre-scale applies: Goldschmidt's coupled
// iteration g -> sqrt(x), h -> 1 / (2 sqrt x) from y = rsq(x), two residual corrections
// g += (x - g^2) h, then the reciprocal of g from 2 h (good to ~2^-44) by one Newton-Raphson
// step and the same correction as div_rn with a = 1. This replaces the v_rcp_f64 and one
// of the two refinement steps that a division takes.
__device__ __forceinline__ void sqrt_and_rcp(double x, double& g, double& r) {
    const double y = __builtin_amdgcn_rsq(x);
    g = x * y;
    double h = 0.5 * y;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    r = 2.0 * h;
    r = __builtin_fma(r, __builtin_fma(-g, r, 1.0), r);
    r = __builtin_fma(__builtin_fma(-g, r, 1.0), r, r);
}

// jacobi_wave::rotation with the short forms, the same bits: every precondition holds when
// d^2 + b^2 is in [2^-40, 2^900). For a Gram of fp32 values summed over at most 2^40 cells,
// |a_ij| < 2^297, and the solve rotates only for |apq| > 1e-6.
__device__ __forceinline__ void jacobi_rotation(double app, double aqq, double apq, double& c, double& s) {
    const double d = aqq - app, b = 2.0 * apq;
    double h, r, ic;  // r = 1 / sqrt(d^2 + b^2), ic = 1 / c
    sqrt_and_rcp(__builtin_fma(d, d, b * b), h, r);
    sqrt_and_rcp(__builtin_fma(0.5 * fabs(d), r, 0.5), c, ic);
    // The correction step rounds wrongly for a divisor whose significand is all ones, and
    // a small angle makes c = 1 - 2^-53 common.
    if (c == 0x1.fffffffffffffp-1) ic = 0x1.0000000000001p0;
    const double sb = d < 0.0 ? -apq : (d > 0.0 ? apq : fabs(apq));
    s = sb * r * ic;
}

}  // namespace slime
