// accept_math.h — the float64 arithmetic of the acceptance weights
// exp(float64(logit - max) / T) (engine/sampling.go:97). Plain functions, so
// that a host compiler can check them against a wider type.
#pragma once

#include <cmath>

namespace yk {

// The temperature as the weights use it: 1 / t rounded, and t for the
// residual of the quotient. Differences below `low` (-1000 t) weigh zero; for
// an infinite temperature there is none, and an overflowed difference makes
// the weight NaN, as -inf / inf is.
struct Temp {
    double t, rt, low;
};

inline Temp make_temp(float temperature) {
    const double t = temperature < 1e300 ? (double)temperature : 1e300;
    return Temp{t, 1.0 / t, temperature < 1e300 ? -1000.0 * t : -HUGE_VAL};
}

// float64(logit - max) / T, correctly rounded down to the double range's
// last few denormals, or -1000 where it is below that.
__device__ __forceinline__ double exponent_of(float l, float mx, const Temp &t) {
    const float d = l - mx;
    double a = (double)d;
    a = a < t.low ? t.low : a;
    const double q = a * t.rt;
    return fma(fma(-q, t.t, a), t.rt, q);
}

// 2^(k/16) as a double and its rounding error.
struct alignas(16) ExpEntry {
    double f, err;
};
__constant__ ExpEntry kExpTab[16] = {
    {0x1.0000000000000p+0, 0x0.0p+0}, {0x1.0b5586cf9890fp+0, 0x1.8a62e4adc610bp-54},
    {0x1.172b83c7d517bp+0, -0x1.19041b9d78a76p-55}, {0x1.2387a6e756238p+0, 0x1.9b07eb6c70573p-54},
    {0x1.306fe0a31b715p+0, 0x1.6f46ad23182e4p-55}, {0x1.3dea64c123422p+0, 0x1.ada0911f09ebcp-55},
    {0x1.4bfdad5362a27p+0, 0x1.d4397afec42e2p-56}, {0x1.5ab07dd485429p+0, 0x1.6324c054647adp-54},
    {0x1.6a09e667f3bcdp+0, -0x1.bdd3413b26456p-54}, {0x1.7a11473eb0187p+0, -0x1.41577ee04992fp-55},
    {0x1.8ace5422aa0dbp+0, 0x1.6e9f156864b27p-54}, {0x1.9c49182a3f090p+0, 0x1.c7c46b071f2bep-56},
    {0x1.ae89f995ad3adp+0, 0x1.7a1cd345dcc81p-54}, {0x1.c199bdd85529cp+0, 0x1.11065895048ddp-55},
    {0x1.d5818dcfba487p+0, 0x1.2ed02d75b3707p-55}, {0x1.ea4afa2a490dap+0, -0x1.e9c23179c2893p-54}};

// exp(x) for -1001 <= x <= 0 (NaN stays NaN): 2^(k/16) from the table (in
// LDS), e^r for r = x - k ln 2 / 16 in two FMA steps (|r| <= ln 2 / 32) by the
// Taylor series to r^7 (remainder below 2e-18). Within 0.58 ulp; a result
// below the normal range rounds twice. The passes that weigh a whole
// vocabulary are bound by its float64 operations (with a plain series to r^13
// the histogram of 144 rows of 151936 took 51 us, with this 45).
__device__ __forceinline__ double exp_nonpos(double x, const ExpEntry *tab) {
    const double k = rint(x * 0x1.71547652b82fep+4);
    const double r = fma(k, -0x1.abc9e3b39803fp-60, fma(k, -0x1.62e42fefa39efp-5, x));
    double p = fma(r, 1.0 / 5040.0, 1.0 / 720.0);
    p = fma(p, r, 1.0 / 120.0);
    p = fma(p, r, 1.0 / 24.0);
    p = fma(p, r, 1.0 / 6.0);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    const int ki = (int)k;
    const ExpEntry f = tab[ki & 15];
    return ldexp(f.f + fma(f.f, p * r, f.err), ki >> 4);
}

// The weight of a valid logit.
__device__ __forceinline__ double soft_weight(float l, float mx, const Temp &t, const ExpEntry *tab) {
    return exp_nonpos(exponent_of(l, mx, t), tab);
}

}  // namespace yk
