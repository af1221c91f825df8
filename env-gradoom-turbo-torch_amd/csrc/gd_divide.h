// 64-bit integer division from float64 arithmetic.  The reciprocal is the caller's, so that the same steps can be run on the host against
// integer division with a reciprocal as far off as the hardware's may be.
#ifndef GD_DIVIDE_H
#define GD_DIVIDE_H

// C truncating division (engine.py:3115-3118), 0 where the divisor is.  gfx950 has no 64-bit integer divider; when both
// magnitudes are below 2^52 the quotient comes from float64 arithmetic.
// The rare large-operand case is a compact shift-subtract loop rather than the compiler's
// unrolled long division, which would be replicated at every call site and push the kernels
// far past the instruction cache.
__device__ __forceinline__ unsigned long long udiv_long(unsigned long long n, unsigned long long d) {
    unsigned long long q = 0, r = 0;
#pragma unroll 1
    for (int i = 63; i >= 0; --i) {
        r = (r << 1) | ((n >> i) & 1);
        if (r >= d) { r -= d; q |= 1ULL << i; }
    }
    return q;
}
template <typename Reciprocal>
__device__ __forceinline__ long long truncated_quotient(long long a, long long b, Reciprocal reciprocal) {
    typedef unsigned long long u64;
    u64 ua = a < 0 ? (u64)0 - (u64)a : (u64)a;
    u64 ub = b < 0 ? (u64)0 - (u64)b : (u64)b;
    if (((ua | ub) >> 52) != 0 || ub == 0) {
        const u64 uq = ub == 0 ? 0 : udiv_long(ua, ub);
        return ((a < 0) != (b < 0)) ? -(long long)uq : (long long)uq;
    }
    // A magnitude under the exponent of 2^52 is that power plus the magnitude, and the other way round.  The reciprocal (off by 2^-24.3
    // of its value at most over 2.1e9 divisors; 2^-22 would do) takes one Newton step, the quotient one step of its own: it is then the
    // true quotient but for one rounding.  That is none where the divisor is one; elsewhere the quotient is below 2^51 and the rounding
    // below an eighth.  Rounded to a whole number it is within 0.7 of the true one, so the quotient or one above.  The remainder, below
    // 2^53, is exact in a fused multiply-add, and its sign tells which.  (With an IEEE division and the library's conversions the chain of
    // 4096 lanes on the 4000-linedef map takes 4.79 ms stage by stage, so 4.76.)
    const double UNIT = 4503599627370496.0;    // 2^52
    const double ad = __builtin_bit_cast(double, ua | 0x4330000000000000ULL) - UNIT, bd = __builtin_bit_cast(double, ub | 0x4330000000000000ULL) - UNIT;
    double r = reciprocal(bd);
    r = __builtin_fma(__builtin_fma(-bd, r, 1.0), r, r);
    double q = ad * r;
    q = __builtin_fma(__builtin_fma(-q, bd, ad), r, q);
    const double whole = q + UNIT;
    const u64 uq = (__builtin_bit_cast(u64, whole) & 0xFFFFFFFFFFFFFULL) - (__builtin_fma(-(whole - UNIT), bd, ad) < 0.0 ? 1u : 0u);
    const u64 sign = (u64)((a ^ b) >> 63);
    return (long long)((uq ^ sign) - sign);
}

#endif
