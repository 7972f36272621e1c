// Correctly rounded FP64 division and square root at a lower price than the compiler's general sequences, for operands of
// ordinary exponents. A division a / b here is Newton's iteration for 1 / b and Markstein's correction of the quotient
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", 1990): q = a y,
// r = a - b q (exact as an fma), q + r y rounds to the quotient; the square root is Goldschmidt's iteration with two
// corrections by the exact residual. What the general sequences add is the scaling of operands near overflow and
// underflow (v_div_scale, v_div_fmas, v_div_fixup, whose condition passes through VCC, so one division waits for the
// other); a caller here checks its operands with plain() and takes the general operators where the check fails, so the
// bits are those of `/` and sqrt() either way. Cycles a wavefront's instruction slot is held, measured on one SIMD:
// a / b 65, divisor() 32 and over() 12; sqrt 88, root() 56.
#pragma once

#include <hip/hip_runtime.h>

namespace luna {

// Whether x's exponent is within [-500, 500]: neither zero, subnormal, infinite, NaN nor near either end of the range.
__device__ __forceinline__ bool plain(double x) {
    constexpr unsigned low = (1023u - 500u) << 20, range = 1001u << 20;
    return ((unsigned)__double2hiint(x) & 0x7fffffffu) - low < range;
}

// b with its correctly rounded reciprocal, for several quotients by the same b.
struct Divisor {
    double b, y;
};
__device__ __forceinline__ Divisor divisor(double b) {
    double y = __builtin_amdgcn_rcp(b);
    y = fma(fma(-b, y, 1.0), y, y);
    y = fma(fma(-b, y, 1.0), y, y);
    return Divisor{b, y};
}
// a / d.b for a plain d.b and an a that is zero or within 2^900 of it either way; a zero quotient is +0 where `/` gives -0
// for a = -0 and d.b > 0.
__device__ __forceinline__ double over(double a, const Divisor& d) {
    const double q = a * d.y;
    return fma(fma(-d.b, q, a), d.y, q);
}

// sqrt(x) of a plain x > 0.
__device__ __forceinline__ double root(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    g = fma(fma(-g, g, x), h, g);
    return g;
}

// round() (half away from zero) in three instructions: |x| plus the largest double below 1/2, truncated.
__device__ __forceinline__ double round_half_away(double x) { return trunc(x + copysign(0.49999999999999994, x)); }

}  // namespace luna
