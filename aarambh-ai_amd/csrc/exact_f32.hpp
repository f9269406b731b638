// Correctly rounded f32 exponentials and quotients without branches, from f64 arithmetic.
// Subnormal results included: at low temperatures most probabilities of a row are subnormal,
// and with exponentials below e^-87 and quotients below 1e-30 left to the plain form nearly
// every wave step runs that as well (28 sequences x 9 rows of 32 000 logits at temperature
// 0.3: 254 us that way, 179 us this way; 207 us with the plain form alone).
// Plain C++ once __device__ and __forceinline__ are defined: the host test includes it.
#pragma once

// (float)exp((double)x) for x in [-inf, 88], or `bad` set: the caller's plain form decides.
// inf is bad, NaN gives 0.  A Taylor polynomial of degree 11 on |r| <= ln 2 / 2, r = x - k ln 2,
// gives e^x within 2^-45 relative (r^12 / 12! is below 2^-47 and the f64 roundings add a few
// 2^-52).  Both ends of a bracket 2^-42 to either side are rounded: where they agree that is
// the value, elsewhere (a midpoint of two f32 values in the bracket, one value in 2^17 or
// fewer) it is bad.  At the clamp, -200, the result is 0 (e^-104 < 2^-150).
__device__ __forceinline__ float expf_fast(float x, bool& bad) {
    const double xd = (double)__builtin_fmaxf(x, -200.0f);
    const double k = __builtin_rint(xd * 1.4426950408889634);
    const double r = __builtin_fma(-k, 0.6931471805599453, xd);
    double p = 1.0 / 39916800.0;
    p = __builtin_fma(p, r, 1.0 / 3628800.0);
    p = __builtin_fma(p, r, 1.0 / 362880.0);
    p = __builtin_fma(p, r, 1.0 / 40320.0);
    p = __builtin_fma(p, r, 1.0 / 5040.0);
    p = __builtin_fma(p, r, 1.0 / 720.0);
    p = __builtin_fma(p, r, 1.0 / 120.0);
    p = __builtin_fma(p, r, 1.0 / 24.0);
    p = __builtin_fma(p, r, 1.0 / 6.0);
    p = __builtin_fma(p, r, 0.5);
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, 1.0);
    const double v = __builtin_ldexp(p, (int)k);
    const float y = (float)__builtin_fma(v, -0x1p-42, v);
    bad = bad | !(y == (float)__builtin_fma(v, 0x1p-42, v));
    return y;
}

// x / d, correctly rounded, with inv = 1 / (double)d.  x * inv in f64 is within 1.5 ulp (of f64) of
// the quotient.  Adding 2 to 4 ulp and clearing the last three bits leaves a value within 7
// ulp, and the quotient itself wherever that has at most 49 bits.  So ties of subnormal results
// (quotients of at most 24 bits) reach the rounding to f32 exactly; any other quotient of two
// 24-bit numbers lies 16 ulp or more from every midpoint of two f32 values.  Infinities, zeros
// and NaN come out as those of x / d.
__device__ __forceinline__ float div_fast(float x, double inv) {
    const double q = (double)x * inv;
    const double up = __builtin_fma(q, 0x1p-51, q);
    return (float)__builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, up) & ~7ull);
}
