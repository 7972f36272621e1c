// The gradient fit's small linear systems (finite_volume.hpp:590-615 Sweep::solve): M = L L^T and M x = b for each variable,
// in the reference's operation order, with the general operators or (Fast) with those of exact_math.hpp, which give the same
// bits where their operands are in range, which FitRange follows; a wavefront whose operands were not solves these systems
// again with the general operators.
#pragma once

#include "exact_math.hpp"

namespace luna {

// The operands of a factor and the solves with it: numerators and divisors.
struct FitRange {
    int numerator = 0;
    Range divisor;
    double size = 0;  // the sum of the solutions' magnitudes: an overflow on the way leaves a NaN in one of them

    __device__ __forceinline__ bool ok() const {
        return numerator > -NUMERATOR && divisor.within(DIVISOR_LEAST, DIVISOR_MOST) && size < 0x1p140;
    }
};

// M's upper triangle to L's lower one; by: L's diagonal as divisors (Fast).
template <int D, bool Fast>
__device__ __forceinline__ void factor(const double (*M)[D + 1], double (*L)[D + 1], Divisor* by, FitRange& range) {
    constexpr int U = D + 1;
#pragma unroll
    for (int p = 0; p < U; ++p)
#pragma unroll
        for (int q = 0; q <= p; ++q) {
            double sum = M[q][p];
#pragma unroll
            for (int m = 0; m < q; ++m) sum -= L[p][m] * L[q][m];
            if constexpr (Fast) {
                if (p == q) {
                    L[p][p] = root(sum);
                    by[p] = divisor(L[p][p]);
                    range.divisor.large(L[p][p]);
                    range.divisor.small(L[p][p]);
                } else {
                    L[p][q] = over(sum, by[q]);
                    range.numerator = min(range.numerator, __builtin_amdgcn_frexp_exp(sum));
                }
            } else {
                L[p][q] = p == q ? sqrt(sum) : sum / L[q][q];
            }
        }
}

template <int D, bool Fast>
__device__ __forceinline__ void solve(const double (*L)[D + 1], const Divisor* by, const double* b, double* x, FitRange& range) {
    constexpr int U = D + 1;
    double z[U];
    const auto quotient = [&](double sum, int p) {
        if constexpr (Fast) {
            range.numerator = min(range.numerator, __builtin_amdgcn_frexp_exp(sum));
            return over(sum, by[p]);
        } else {
            return sum / L[p][p];
        }
    };
#pragma unroll
    for (int p = 0; p < U; ++p) {
        double sum = b[p];
#pragma unroll
        for (int m = 0; m < p; ++m) sum -= L[p][m] * z[m];
        z[p] = quotient(sum, p);
    }
#pragma unroll
    for (int p = U - 1; p >= 0; --p) {
        double sum = z[p];
#pragma unroll
        for (int m = p + 1; m < U; ++m) sum -= L[m][p] * x[m];
        x[p] = quotient(sum, p);
        if constexpr (Fast) range.size += fabs(x[p]);
    }
}

}  // namespace luna
