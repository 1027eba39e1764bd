/*
 * hd_fastdiv.h -- several FP64 quotients from one refined reciprocal, with
 * the bits of the division operator (gfx950 device code).
 *
 * The correctly rounded division n / e is computed on this part as
 *   y0 = rcp(e), two Newton steps y -> y + y (1 - e y), q0 = n y,
 *   r = n - e q0 (one FMA, exact), q = q0 + r y (one FMA),
 * (the last two steps are Markstein's correction of a quotient, P. Markstein,
 * IBM J. Res. Dev. 34, 1990, with y accurate to about a rounding of 1 / e and
 * r exact), around which it scales operands that are near the ends of the
 * exponent range and repairs zeros, infinities and NaNs.
 * Every operation in the middle is invariant under scaling by powers of two,
 * so wherever nothing overflows or underflows, leaving the scaling out changes
 * no bit; and y depends on e alone, so quotients by the same e share it (75
 * cycles for a division, about 45 for y and 20 for each quotient, the part's
 * measured latencies).  The two cases that differ are kept out by the caller:
 *  - a numerator of -0 over e > 0 would give +0 (quot; quot_pos gives the
 *    right zeros for every numerator while e > 0);
 *  - operands out of range: Range collects the exponents of divisors and
 *    numerators (zero, infinity and NaN count as exponent 0: zeros are
 *    right, and an infinity or NaN, a zero divisor or an overflow leaves a
 *    NaN or infinity in the result, which the caller tests for).
 */
#ifndef HD_FASTDIV_H
#define HD_FASTDIV_H

#include <hip/hip_runtime.h>

namespace hd_div {

__device__ __forceinline__ double rcp_refined(double e)
{
    double y = __builtin_amdgcn_rcp(e);
    y = fma(y, fma(-e, y, 1.0), y);
    return fma(y, fma(-e, y, 1.0), y);
}

/* n / e, y = rcp_refined(e); n not -0 unless e < 0 */
__device__ __forceinline__ double quot(double n, double e, double y)
{
    const double q = n * y;
    return fma(fma(-e, q, n), y, q);
}

/* n / e for e > 0, any zero n */
__device__ __forceinline__ double quot_pos(double n, double e, double y)
{
    const double q = n * y;
    return fma(-fma(e, q, -n), y, q);
}

__device__ __forceinline__ bool neg_zero(double v) { return __builtin_amdgcn_class(v, 0x20); }
__device__ __forceinline__ bool finite(double v) { return fabs(v) <= 1.7976931348623157e308; }

/* Exponents seen: the smallest of the numerators (or of whatever num is
 * given), both ends of the divisors.  With divisors in 2^[-100, 100] and a
 * numerator of at least 2^-900 (or zero) every intermediate, down to the
 * remainder's last bit 2^-106 below the numerator, is a normal number or
 * exact. */
struct Range {
    int lo = 0, dlo = 0, dhi = 0;
    __device__ __forceinline__ void den(double e)
    {
        const int x = __builtin_amdgcn_frexp_exp(e);
        dlo = x < dlo ? x : dlo;
        dhi = x > dhi ? x : dhi;
    }
    __device__ __forceinline__ void num(double n)
    {
        const int x = __builtin_amdgcn_frexp_exp(n);
        lo = x < lo ? x : lo;
    }
    __device__ __forceinline__ bool den_ok() const { return dlo >= -100 && dhi <= 100; }
    __device__ __forceinline__ bool ok() const { return lo >= -900 && den_ok(); }
};

} // namespace hd_div

#endif
