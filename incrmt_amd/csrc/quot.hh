// Quotients by a divisor whose reciprocal is kept: five dependent operations
// instead of a division's thirty.
#ifndef INCRMT_QUOT_HH
#define INCRMT_QUOT_HH

#ifndef __HIPCC__
#ifndef __host__
#define __host__
#define __device__
#endif
#endif
#include <cstring>

namespace incrmt {

// n / d from y = 1 / d correctly rounded (P. Markstein, IBM J. Res. Dev. 34,
// 1990: with q within a rounding of n / d, the remainder n - d q is exact in one
// fused operation and q + y (n - d q) rounds to the quotient; the first
// correction brings q there). These are the division's bits for
// quot_divisor(d) and quot_numerator(n), where neither the quotient nor the
// remainder, down to 2^-47 (2^-106) of n, leaves the normal numbers. Other finite
// n (the right-hand side of a single-precision cycle is an unscaled residual,
// so n may be tiny) give a finite quotient to one unit in its last place, since a
// remainder may underflow; an infinite n or quotient gives NaN where a
// division gives infinity. Testing each n, and repeating such a cycle with
// divisions, makes a cycle of a 32^2 MAC solve 26.9 us instead of 25.5, of a
// 33^2 FEM solve 39.0 instead of 36.2 (double precision). POS, the sign of d,
// decides the form that keeps the sign of a zero.
__host__ __device__ inline double quot_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__host__ __device__ inline float quot_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <bool POS, class T>
__host__ __device__ inline T quot(T n, T d, T y) {
    T q = n * y;
    q = POS ? quot_fma(-quot_fma(d, q, -n), y, q) : quot_fma(quot_fma(-d, q, n), y, q);
    return POS ? quot_fma(-quot_fma(d, q, -n), y, q) : quot_fma(quot_fma(-d, q, n), y, q);
}

// 2^-E <= |v| < 2^E, from the exponent bits
template <int E>
__host__ __device__ inline bool within_2to(double v) {
    unsigned long long b;
    memcpy(&b, &v, sizeof b);
    return ((unsigned)(b >> 32) & 0x7fffffffu) - ((1023u - E) << 20) < 2u * E << 20;
}
template <int E>
__host__ __device__ inline bool within_2to(float v) {
    unsigned b;
    memcpy(&b, &v, sizeof b);
    return (b & 0x7fffffffu) - ((127u - E) << 23) < 2u * E << 23;
}
template <bool POS>
__host__ __device__ inline bool quot_divisor(double d) { return within_2to<400>(d) && (d > 0) == POS; }
template <bool POS>
__host__ __device__ inline bool quot_divisor(float d) { return within_2to<40>(d) && (d > 0) == POS; }
__host__ __device__ inline bool quot_numerator(double n) { return within_2to<400>(n) | (n == 0); }
__host__ __device__ inline bool quot_numerator(float n) { return within_2to<80>(n) | (n == 0); }

}  // namespace incrmt

#endif
