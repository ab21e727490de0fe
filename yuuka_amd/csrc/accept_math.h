// accept_math.h — the float64 arithmetic of the acceptance weights
// exp(float64(logit - max) / T) (engine/sampling.go:97). Plain functions, so
// that a host compiler can check them against a wider type.
#pragma once

#include <cmath>
#include <cstdint>

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

// Members of a boundary tie group (weight w each) that top_p keeps: they join
// one by one, as the sampler's running sum adds their shares
// (sampling.go:107-113), from the weight `before` ahead of the group: the
// first i with cum_i >= top_p, at most `ties`. Once two sums of a binade
// follow each other, each further one in it rises by the same multiple of its
// last place (a share that lies halfway between two multiples rounds to even,
// and even sums stay even), so all but the binade's last steps are taken at
// once and exactly. (One addition after the other, 93750 equal logits took a
// thread 4.6 ms.)
__device__ __forceinline__ uint32_t tie_members(double before, double w, double total, double top_p, uint32_t ties) {
    const double q = w / total;
    double cum = before / total, top = 0.0;  // top: the end of the sum's binade
    int inside = 0;                          // sums in it so far
    for (uint32_t i = 1; i < ties; i++) {
        double next = cum + q;
        if (next >= top_p) return i;
        if (!(next > cum)) return ties;  // no share, or one too small to count
        if (next < top) {
            inside++;
        } else {
            top = ldexp(1.0, ilogb(next) + 1);
            inside = 1;
        }
        if (inside >= 3) {
            const double step = next - cum, room = (fmin(top, top_p) - next) / step - 2.0;
            if (room >= 1.0) {
                const uint32_t skip = room < (double)(ties - 1 - i) ? (uint32_t)room : ties - 1 - i;
                next += (double)skip * step;
                i += skip;
            }
        }
        cum = next;
    }
    return ties;
}

}  // namespace yk
