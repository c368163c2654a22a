// Quotients s / d from the correctly rounded reciprocal ri = 1 / d, on chains where a division's latency counts.
// Host code may include this as well.
#pragma once

#include <cmath>

#ifdef __HIPCC__
#define PFEM_HD __host__ __device__ __forceinline__
#else
#define PFEM_HD inline
#endif

namespace pfem {

// The first quotient is within two units in the last place, the second within one, and Markstein's theorem ("IA-64
// and Elementary Functions", 2000) makes the third the correctly rounded one as long as no step under- or
// overflows: |d| in [2^-100, 2^100] (else ri is stored as a NaN) and |q| >= 2^-800 or s = 0. A result outside (NaNs
// included) is formed again by the division.
PFEM_HD double quotient(double s, double d, double ri)
{
    const double q0 = s * ri;
    const double q1 = __builtin_fma(__builtin_fma(-d, q0, s), ri, q0);
    return __builtin_copysign(__builtin_fma(__builtin_fma(-d, q1, s), ri, q1), q0);   // (the sign of a zero)
}
PFEM_HD bool quotient_ok(double q) { return __builtin_fabs(q) >= 0x1p-800 || q == 0.0; }
PFEM_HD float quotient(float s, float d, double) { return s / d; }
PFEM_HD bool quotient_ok(float q) { return q == q; }

// One correction: within one unit in the last place (the division's value in each of 4e8 random operands). Where the
// correction has no value (an infinite quotient, a zero divisor) the uncorrected quotient, as the division has it.
PFEM_HD double quotient_near(double s, double d, double ri)
{
    const double q0 = s * ri;
    const double q1 = __builtin_fma(__builtin_fma(-q0, d, s), ri, q0);
    return q1 == q1 ? q1 : q0;
}

}  // namespace pfem
