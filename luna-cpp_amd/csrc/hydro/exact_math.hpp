// Correctly rounded FP64 division and square root at a lower price than the compiler's general sequences, for operands of
// ordinary exponents. A division a / b here is Newton's iteration for 1 / b and Markstein's correction of the quotient
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", 1990): q = a y,
// r = a - b q (exact as an fma), q + r y rounds to the quotient; the square root is Goldschmidt's iteration with two
// corrections by the exact residual. What the general sequences add is the scaling of operands near overflow and
// underflow (v_div_scale, v_div_fmas, v_div_fixup, whose condition passes through VCC, so one division waits for the
// other); a caller here checks its operands (Range) and takes the general operators where a check fails, so the bits are
// those of `/` and sqrt() either way. Cycles a wavefront's instruction slot is held, measured on one SIMD: a / b 65, divisor()
// 32 and over() 12; sqrt 88, root() 56.
// What the ranges have to keep: over()'s residual a - b q is a multiple of 2^(e(a) - 106), so it is exact for |a| >= 2^-968
// (measured, 10^6 numerators of each exponent: the first quotients off in the last bit at 2^-1000), root()'s likewise; q
// has to be normal; and 1 / b may be neither subnormal nor infinite.
#pragma once

#include <hip/hip_runtime.h>

namespace luna {

// Whether a run of operands was in range, followed by the largest high word and the smallest exponents instead of a test
// each (two to four instructions without a wait for a mask, where a test of the range is four with one).
struct Range {
    int top = 0;             // the largest high word of those that may not be too large: negative ones never are
    unsigned bottom = ~0u;   // the smallest high word of those that may be neither too small nor zero
    int exponent = 0;        // the smallest exponent of those that may be zero (frexp's: 0 for a zero, an infinity or a NaN)

    static constexpr int high(int exponent) { return (1023 + exponent) << 20; }
    __device__ __forceinline__ void large(double x) { top = max(top, __double2hiint(x)); }
    __device__ __forceinline__ void small(double x) { bottom = min(bottom, (unsigned)__double2hiint(x)); }
    __device__ __forceinline__ void small_or_zero(double x) { exponent = min(exponent, __builtin_amdgcn_frexp_exp(x)); }
    // All of them within 2^-least .. 2^most.
    __device__ __forceinline__ bool within(int least, int most) const {
        return top < high(most) && bottom >= (unsigned)high(-least) && exponent > -least;
    }
};

// over(a, d) is the quotient for numerators that are zero or at least 2^-NUMERATOR (an infinite, NaN or too large one leaves
// an infinite or NaN quotient) and divisors from 2^-DIVISOR_LEAST to 2^DIVISOR_MOST, whose squares are in root()'s range: then
// neither the quotient nor the residual falls below the normal numbers.
constexpr int NUMERATOR = 750, DIVISOR_LEAST = 450, DIVISOR_MOST = 250;

// b with its reciprocal, for several quotients by the same b. The reciprocal is the correctly rounded one but for a few b
// whose significand is within 13 ulps of 2; over()'s quotients are right for those too (every b within 4096 ulps of 2 and of 1,
// each with 16384 numerators).
struct Divisor {
    double b, y;
};
__device__ __forceinline__ Divisor divisor(double b) {
    double y = __builtin_amdgcn_rcp(b);
    y = fma(fma(-b, y, 1.0), y, y);
    y = fma(fma(-b, y, 1.0), y, y);
    return Divisor{b, y};
}
// a / d.b where a and d.b are in range; a zero quotient is +0 where `/` gives -0 for a = -0 and d.b > 0.
__device__ __forceinline__ double over(double a, const Divisor& d) {
    const double q = a * d.y;
    return fma(fma(-d.b, q, a), d.y, q);
}

// sqrt(x) for x from 2^-900 to 2^1000.
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
